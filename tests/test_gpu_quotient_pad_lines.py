"""Fibonacci quotient and zero pad on both sides of the sizes from which a thread takes
four words, at any alignment and ragged ends, against numpy. Runs on the MI355X."""

import ctypes as C

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


@pytest.mark.parametrize("shift", [0, 1, 3])
@pytest.mark.parametrize("n", [(1 << 18) - 1, 1 << 18, (1 << 18) + 1, (1 << 18) + 3, (1 << 19) + 2])
def test_quotient(vx, n, shift):
    rng = np.random.default_rng(n)
    t = rng.integers(0, P, n, dtype=np.int64)
    alpha = rng.integers(0, P, 4, dtype=np.int64)
    dt = vx.DeviceBuffer.from_host(np.concatenate([np.zeros(shift, np.int64), t]).astype(np.uint32))
    d = (np.roll(t, -2) - np.roll(t, -1) - t) % P
    for off, chunk in ((0, n), (n - (1 << 18) if n > 1 << 18 else 5, min(1 << 18, n - 5))):
        out = [vx.DeviceBuffer.from_host(np.full(chunk + shift + 1, 0xFFFFFFFF, np.uint32)) for _ in range(4)]
        vx.lib.cuda_fibonacci_quotient_chunk(dt.addr + 4 * shift, *[o.addr + 4 * shift for o in out],
                                             (C.c_uint32 * 4)(*[int(a) for a in alpha]), off, chunk, n)
        vx.synchronize()
        vx.check()
        for c in range(4):
            got = out[c].to_host()
            assert np.array_equal(got[shift:-1], (d * alpha[c] % P)[off:off + chunk].astype(np.uint32))
            assert got[-1] == 0xFFFFFFFF and (got[:shift] == 0xFFFFFFFF).all()


@pytest.mark.parametrize("shift", [0, 2])
@pytest.mark.parametrize("n,m", [(1 << 17, (1 << 19) - 1), (1 << 17, 1 << 19), ((1 << 17) + 1, (1 << 19) + 3),
                                 ((1 << 19) + 5, (1 << 19) + 5), (1, 1 << 19)])
def test_pad(vx, n, m, shift):
    t = np.random.default_rng(n).integers(0, P, n, dtype=np.int64).astype(np.uint32)
    src = vx.DeviceBuffer.from_host(np.concatenate([np.zeros(shift, np.uint32), t]))
    dst = vx.DeviceBuffer.from_host(np.full(m + shift + 1, 0xFFFFFFFF, np.uint32))
    vx.lib.cuda_zero_pad(src.addr + 4 * shift, dst.addr + 4 * shift, n, m)
    vx.synchronize()
    vx.check()
    got = dst.to_host()
    assert np.array_equal(got[shift:-1], np.concatenate([t, np.zeros(m - n, np.uint32)]))
    assert got[-1] == 0xFFFFFFFF and (got[:shift] == 0xFFFFFFFF).all()
