"""Default splits of blowup-4 evaluations: the rule on the CPU; proofs at the sizes
where the number of passes or their segments change, with the general table and
back, against the oracle."""

import os
import subprocess

import pytest

import oracle_lib as O

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rule(tmp_path):
    exe = tmp_path / "lde_plan_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(HERE, "host", "lde_plan_test.cpp"), "-o", str(exe)], check=True)
    assert "lde plans: ok" in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


@pytest.mark.gpu
@pytest.mark.parametrize("log_n", [10, 11, 12, 13, 15, 16, 20])
def test_proofs_with_default_plans(vx, log_n):
    k, exp = log_n + 2, O.prove(5, 9, log_n)
    vx.lib.vx_ntt_plan_reset()
    try:
        plan = vx.ntt_lde_plan(k)
        assert plan[-1][2] == (1 if k > 12 else 0)
        assert vx.prove(5, 9, log_n) == exp
        vx.ntt_lde_plan_set(k, [])  # the general table
        assert vx.ntt_lde_plan(k) == [(m, c, 0) for m, c in vx.ntt_plan(k)]
        assert vx.prove(5, 9, log_n) == exp
        vx.lib.vx_ntt_plan_reset()
        assert vx.ntt_lde_plan(k) == plan
        m = min(k - 6, 13)
        general = [(m, 0), (k - m, 5)]  # a general plan of the size serves its evaluations too
        vx.ntt_plan_set(k, general)
        assert vx.ntt_lde_plan(k) == [(m, c, 0) for m, c in vx.ntt_plan(k)]
        assert vx.prove(5, 9, log_n) == exp
    finally:
        vx.lib.vx_ntt_plan_reset()
