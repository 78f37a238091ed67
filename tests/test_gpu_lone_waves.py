"""Hash launches on both sides of one wave a SIMD (2^16 threads), where the
compression changes its issue priorities, against the oracle. Runs on the MI355X."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1
LONE = 1 << 16


def rnd(seed, n):
    return np.random.default_rng(seed).integers(0, P, n, dtype=np.uint64).astype(np.uint32)


def device_columns(vx, cols):
    bufs = [vx.DeviceBuffer.from_host(c) for c in cols]
    return bufs, vx.DeviceBuffer.from_host(np.array([b.addr for b in bufs], np.uint64).view(np.uint32))


@pytest.mark.parametrize("n_cols", [1, 3, 4, 16])
@pytest.mark.parametrize("n", [1, LONE - 1, LONE, LONE + 1])
def test_hash_leaves(vx, n_cols, n):
    cols = [rnd(31 * n_cols + c, n) for c in range(n_cols)]
    bufs, ptrs = device_columns(vx, cols)
    out = vx.DeviceBuffer(8 * n)
    vx.lib.cuda_merkle_hash_leaves(ptrs.addr, out.addr, n_cols, n)
    vx.synchronize()
    assert np.array_equal(out.to_host(), O.leaf_hashes(cols))


@pytest.mark.parametrize("n", [2, 2 * LONE - 2, 2 * LONE, 2 * LONE + 2])
def test_merge(vx, n):
    cols = [rnd(77 + c, n) for c in range(4)]
    bufs, _ = device_columns(vx, cols)
    par = vx.DeviceBuffer(4 * n)
    vx.lib.cuda_merkle_hash_leaves_merge_soa4(*[b.addr for b in bufs], par.addr, n)
    vx.synchronize()
    leaves, want = O.leaf_hashes(cols), np.zeros(4 * n, np.uint32)
    O.lib().orc_merkle_node_layer(leaves.ctypes.data, n // 2, want.ctypes.data)
    assert np.array_equal(par.to_host(), want)


# the tail kernel's first level: nodes copied (16), read in place by quads (256), by lanes
# (512 items are 256 parents, one wave a SIMD)
@pytest.mark.parametrize("n", [1, 2, 4, 8, 16, 32, 256, 512, 1024, 2048])
def test_roots(vx, n):
    nodes = rnd(5 + n, 8 * n)
    buf, root = vx.DeviceBuffer.from_host(nodes), vx.DeviceBuffer(8)
    vx.lib.cuda_merkle_reduce_to_root(buf.addr, root.addr, n)
    level = nodes
    while len(level) > 8:
        up = np.zeros(len(level) // 2, np.uint32)
        O.lib().orc_merkle_node_layer(level.ctypes.data, len(up) // 8, up.ctypes.data)
        level = up
    vx.synchronize()
    assert np.array_equal(root.to_host(), level)
    if n > 1:
        cols = [rnd(9 + c, n) for c in range(4)]
        bufs, _ = device_columns(vx, cols)
        vx.lib.cuda_merkle_commit_small_soa4(*[b.addr for b in bufs], root.addr, n)
        vx.synchronize()
        assert np.array_equal(root.to_host(), O.merkle_root(cols))
