"""Folds, quotient and zero pad of the kernel ABI at ragged sizes and on
pointers that allow 16-byte accesses or not, against the oracle; challenges with
zero coordinates. Runs on the MI355X."""

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


def rnd(seed, n):
    return np.random.default_rng(seed).integers(0, P, n, dtype=np.uint64).astype(np.uint32)


def h32(vals):
    return (C.c_uint32 * len(vals))(*[int(v) for v in vals])


class Words:
    """n device words `shift` words past a 256-byte aligned address."""

    def __init__(self, vx, host, shift):
        self.shift, self.n = shift, len(host)
        self.buf = vx.DeviceBuffer.from_host(np.concatenate([np.zeros(shift, np.uint32), host]))
        self.addr = self.buf.addr + 4 * shift

    def get(self):
        return self.buf.to_host()[self.shift:]


ALPHAS = [[5, 7, 11, 13], [0, 0, 0, 0], [P - 1, 0, P - 1, 1], [0, P - 1, P - 1, P - 1]]


@pytest.mark.parametrize("shift", [0, 1, 2])
@pytest.mark.parametrize("half", [1, 2, 3, 255, 512, 513, 1021])
def test_folds(vx, half, shift):
    for k, alpha in enumerate(ALPHAS):
        cols = [rnd(10 * half + c + k, 2 * half) for c in range(4)]
        cols[0][:2] = [P - 1, 0]
        tw, prev, sq = rnd(7 + half, half), [rnd(99 + c, half) for c in range(4)], rnd(3 + k, 4)
        src = [Words(vx, c, shift) for c in cols]
        dtw, dst = Words(vx, tw, shift), [Words(vx, np.zeros(half, np.uint32), shift) for _ in range(4)]
        vx.lib.cuda_fold_line_soa(*[s.addr for s in src], dtw.addr, *[d.addr for d in dst], h32(alpha), half)
        want = O.fold_line(cols, tw, alpha)
        vx.synchronize()
        assert np.array_equal(np.stack([d.get() for d in dst]), np.asarray(want).reshape(4, half))
        onto = [Words(vx, p, shift) for p in prev]
        vx.lib.cuda_fold_circle_into_line_soa(*[d.addr for d in onto], *[s.addr for s in src], dtw.addr, h32(alpha),
                                              h32(sq), half)
        vx.synchronize()
        got = np.stack([d.get() for d in onto])
        for i in {0, half // 2, half - 1}:
            exp = (C.c_uint32 * 4)()
            O.lib().orc_qm31_mul(h32([p[i] for p in prev]), h32(sq), exp)
            fold = np.asarray(want).reshape(4, half)[:, i]
            assert [int(x) for x in got[:, i]] == [(int(e) + int(f)) % P for e, f in zip(exp, fold)]
    vx.check()


@pytest.mark.parametrize("shift", [0, 3])
@pytest.mark.parametrize("n", [1, 2, 3, 7, 8, 9, 1023, 1024, 1030])
def test_quotient_and_pad(vx, n, shift):
    t, alpha = rnd(n, n), rnd(n + 1, 4)
    dt = Words(vx, t, shift)
    for off, chunk in {(0, n), (n // 2, n - n // 2), (min(4, n - 1), 1)}:
        out = [Words(vx, np.zeros(chunk, np.uint32), shift) for _ in range(4)]
        vx.lib.cuda_fibonacci_quotient_chunk(dt.addr, *[o.addr for o in out], h32(alpha), off, chunk, n)
        vx.synchronize()
        x = t.astype(np.int64)
        d = (np.roll(x, -2) - np.roll(x, -1) - x) % P
        for c in range(4):
            assert np.array_equal(out[c].get(), (d * int(alpha[c]) % P)[off:off + chunk].astype(np.uint32))
    for m in (n, n + 1, n + 3, 4 * n):
        dst = Words(vx, np.full(m, 0xFFFFFFFF, np.uint32), shift)
        vx.lib.cuda_zero_pad(dt.addr, dst.addr, n, m)
        vx.synchronize()
        assert np.array_equal(dst.get(), np.concatenate([t, np.zeros(m - n, np.uint32)]))
    vx.check()
