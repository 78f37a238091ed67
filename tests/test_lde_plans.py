"""Splits of sizes without a plan: the rules on the CPU; transforms on both sides of
the general one's line; proofs at the sizes
where the number of passes or their segments change, with the general table and
back, against the oracle."""

import ctypes as C
import os
import subprocess

import numpy as np
import pytest

import oracle_lib as O

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rule(tmp_path):
    exe = tmp_path / "lde_plan_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(HERE, "host", "lde_plan_test.cpp"), "-o", str(exe)], check=True)
    assert "lde plans: ok" in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


@pytest.mark.gpu
@pytest.mark.parametrize("k", [19, 20, 21, 22, 23])
def test_transforms_without_a_plan(vx, k):
    """A batch of two columns forward against the oracle, and back."""
    n = 1 << k
    vx.lib.vx_ntt_plan_reset()
    line, circle, iline, icircle, offs, sizes = O.ntt_twiddles(1, k)
    cols = [np.random.default_rng(10 * k + c).integers(0, (1 << 31) - 1, n, dtype=np.uint32) for c in range(2)]
    tabs = [vx.DeviceBuffer.from_host(a) for a in (line, circle, iline, icircle)]
    bufs = [vx.DeviceBuffer.from_host(c) for c in cols]
    ptrs = vx.DeviceBuffer.from_host(np.array([b.addr for b in bufs], np.uint64).view(np.uint32))
    ho, hs = ((C.c_uint32 * (k - 1))(*[int(v) for v in a[: k - 1]]) for a in (offs, sizes))
    vx.lib.cuda_circle_ntt_evaluate_batch(ptrs.ptr, tabs[0].ptr, tabs[1].ptr, ho, hs, k - 1, n, 2)
    for b, c in zip(bufs, cols):
        exp = c.copy()
        O.lib().orc_ntt_evaluate(exp.ctypes.data, line.ctypes.data, circle.ctypes.data, k)
        assert np.array_equal(b.to_host(), exp)
    vx.lib.cuda_circle_ntt_interpolate_batch(ptrs.ptr, tabs[2].ptr, tabs[3].ptr, ho, hs, k - 1, n, 2)
    for b, c in zip(bufs, cols):
        assert np.array_equal(b.to_host(), c)
    vx.check()


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
