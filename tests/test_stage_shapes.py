"""Stage shapes of the Merkle engine: the rule itself on the CPU, and proofs and
wide roots at launch sizes on both sides of its lines against the oracle."""

import os
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from inputs import m31_columns

HERE = os.path.dirname(os.path.abspath(__file__))


def test_rule(tmp_path):
    exe = tmp_path / "stage_shape_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(HERE, "host", "stage_shape_test.cpp"), "-o", str(exe)], check=True)
    assert "stage shapes: ok" in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


# launches of 2^17 .. 2^22 leaves, as one proof and as batches
@pytest.mark.gpu
@pytest.mark.parametrize("log_n,count", [(15, 1), (16, 1), (17, 1), (18, 1), (20, 1), (11, 16), (10, 65), (13, 33), (15, 32)])
def test_proofs_at_every_shape(vx, log_n, count):
    ab = [(7 + 3 * i, 1000 + i * i) for i in range(count)]
    p = vx.Prover(log_n, capacity=count)
    got = p.prove_batch(ab)
    p.close()
    for i in sorted({0, count // 2, count - 1}):
        assert got[i] == O.prove(*ab[i], log_n), f"proof {i}"


@pytest.mark.gpu
@pytest.mark.parametrize("logs", [[5, 16], [3, 7, 7, 7, 17], [14] * 2 + [18] * 17])
def test_wide_at_every_shape(vx, logs):
    cols = m31_columns(11, logs)
    w = vx.WideCommit(logs, 2, 3)
    bufs = [vx.DeviceBuffer.from_host(c) for c in cols]
    w.commit_device([b.addr for b in bufs])
    got = w.results()
    exp = O.wide_commit(cols, logs, 2, 3)
    for g, e in zip(got, exp):
        assert np.array_equal(g, e)
    w.close()
