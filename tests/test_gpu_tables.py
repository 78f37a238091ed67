"""Tile roots and node levels on both sides of the switches of the work per tile, fold-twiddle
sources and traces at run and block edges, batch inverses of every words-per-thread count:
against the oracle. Runs on the MI355X."""

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


def rnd(seed, n):
    return np.random.default_rng(seed).integers(0, P, n, dtype=np.uint64).astype(np.uint32)


@pytest.mark.parametrize("soa4,n_cols", [(True, 4), (False, 1), (False, 4), (False, 3), (False, 17)])
@pytest.mark.parametrize("tiles,rest", [(1, 0), (3, 512), (256, 6), (257, 0), (4095, 0), (4099, 0)])
def test_tile_roots(vx, soa4, n_cols, tiles, rest):
    n = 1024 * tiles + rest
    base = rnd(1, n + 64)
    cols = [base[c: c + n] for c in range(n_cols)]
    bufs = [vx.DeviceBuffer.from_host(np.ascontiguousarray(c)) for c in cols]
    out = vx.DeviceBuffer.from_host(np.full(8 * tiles + 8, 7, np.uint32))
    if soa4:
        vx.lib.cuda_merkle_tiled_soa4(*[b.ptr for b in bufs], out.ptr, n)
    else:
        ptrs = vx.DeviceBuffer.from_host(np.array([b.addr for b in bufs], np.uint64).view(np.uint32))
        vx.lib.cuda_merkle_tiled_generic(ptrs.ptr, out.ptr, n_cols, n)
    vx.synchronize()
    got = out.to_host()
    assert (got[8 * tiles:] == 7).all()
    picks = sorted({0, 1, 7, 8, tiles // 2, tiles - 2, tiles - 1} & set(range(tiles)))
    for t in picks:
        exp = O.merkle_root([np.ascontiguousarray(c[1024 * t: 1024 * (t + 1)]) for c in cols])
        assert np.array_equal(got[8 * t: 8 * t + 8], exp), t
    vx.check()


def mul(a, b):
    return (a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P


def power(p, e):
    r = (1, 0)
    while e:
        if e & 1:
            r = mul(r, p)
        p, e = mul(p, p), e >> 1
    return r


def brev(x, bits):
    return int(format(x, "b").zfill(bits)[::-1], 2) if bits else 0


@pytest.mark.parametrize("use_y", [0, 1])
@pytest.mark.parametrize("log_n,n", [(1, 2), (2, 4), (4, 16), (5, 32), (6, 64), (13, 1 << 13), (14, 1 << 14),
                                     (20, 1 << 20), (20, 1000), (3, 64)])
def test_fold_sources(vx, log_n, n, use_y):
    g = (2, 1268011823)
    initial, step = power(g, 12345), power(g, 1 << (31 - log_n))
    out = vx.DeviceBuffer.from_host(np.full(n // 2 + 1, 7, np.uint32))
    vx.lib.cuda_compute_fold_twiddle_sources(*initial, *step, out.ptr, n, log_n, use_y)
    vx.synchronize()
    got = out.to_host()
    assert got[n // 2] == 7
    half = n // 2
    picks = range(half) if half <= 512 else sorted(set(rnd(5, 300) % half) | {0, 15, 16, 1023, 1024, 4095, half - 1})
    for i in picks:
        e = brev((2 * int(i)) & ((1 << log_n) - 1), log_n)
        assert got[i] == mul(initial, power(step, e))[use_y], i
    vx.check()


@pytest.mark.parametrize("n", [1, 3, 4, 5, 63, 64, 65, 513, (1 << 20) - 1, 1 << 20, (1 << 20) + 3, (1 << 22) - 1,
                               1 << 22, (1 << 22) + 77])
def test_batch_inverse(vx, n):
    v = rnd(9, n)
    v[rnd(10, max(1, n // 50)) % n] = 0
    src, dst = vx.DeviceBuffer.from_host(v), vx.DeviceBuffer(n)
    vx.lib.cuda_batch_inverse_m31(src.ptr, dst.ptr, n)
    vx.synchronize()
    got = dst.to_host().astype(np.uint64)
    live = np.repeat(v[::64] != 0, 64)[:n] & (v != 0)
    assert (got[~live] == 0).all()
    assert (got[live] * v[live] % P == 1).all() and (got < P).all()
    vx.check()


@pytest.mark.parametrize("log_n", [1, 2, 3, 4, 5, 11, 12, 13, 20])
@pytest.mark.parametrize("a,b", [(1, 1), (0, P - 1), (P - 1, 12345)])
def test_fibonacci_trace(vx, log_n, a, b):
    n = 1 << log_n
    out = vx.DeviceBuffer.from_host(np.full(n + 2, 7, np.uint32))
    vx.lib.vx_fibonacci_trace(a, b, log_n, C.c_void_p(out.addr + 4), None)
    vx.synchronize()
    got = out.to_host()
    assert got[0] == 7 and got[n + 1] == 7
    assert np.array_equal(got[1: n + 1], O.fibonacci_trace(a, b, log_n))
    vx.check()


@pytest.mark.parametrize("n", [1, 2, 3, 63, 65, 1 << 14, (1 << 14) + 1, 1 << 16, (1 << 16) + 5])
def test_hash_nodes(vx, n):
    ch = np.random.default_rng(n).integers(0, 1 << 32, 16 * n, dtype=np.uint64).astype(np.uint32)
    src, dst = vx.DeviceBuffer.from_host(ch), vx.DeviceBuffer.from_host(np.full(8 * n + 1, 7, np.uint32))
    vx.lib.cuda_merkle_hash_nodes(src.ptr, dst.ptr, n)
    vx.synchronize()
    exp = np.zeros(8 * n, np.uint32)
    O.lib().orc_merkle_node_layer(ch.ctypes.data, n, exp.ctypes.data)
    got = dst.to_host()
    assert np.array_equal(got[:-1], exp) and got[-1] == 7
    vx.check()
