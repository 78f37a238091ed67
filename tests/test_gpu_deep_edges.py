"""DEEP kernels on both sides of the lines where a thread takes more rows, with
every remainder of the column groups and the largest canonical values, against
the oracle. Runs on the MI355X."""

import numpy as np
import pytest

import oracle_lib as O
from test_gpu_deep import gpu_combine, gpu_numerators, oracle_pipeline, rnd

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


@pytest.mark.parametrize("L", [9, 17, 18])
@pytest.mark.parametrize("n_points,n_cols", [(1, 4), (2, 5), (3, 6), (4, 7), (4, 8), (2, 3)])
def test_fused_rows_and_remainders(vx, L, n_points, n_cols):
    rng = np.random.default_rng(L + 10 * n_points + n_cols)
    logs = [L - 2] * (n_cols // 2) + [L] * (n_cols - n_cols // 2)
    cols = [rnd(rng, 1 << l) for l in logs]
    cols[0][:] = P - 1
    cols[-1][: 1 << (L - 1)] = P - 1
    points, lc = rnd(rng, n_points, 8), rnd(rng, n_points, n_cols, 12)
    lc[0] = P - 1
    dxs, dys = vx.circle_domain_points(L)
    bufs, outs = [vx.DeviceBuffer.from_host(c) for c in cols], [vx.DeviceBuffer(1 << L) for _ in range(4)]
    dq = vx.DeepQuotient(n_cols, n_points)
    dq.quotient([b.addr for b in bufs], logs, points, lc, L, dxs.addr, dys.addr, [o.addr for o in outs])
    vx.synchronize()
    dq.close()
    exp = oracle_pipeline(cols, logs, points, lc, L, *O.circle_domain_brev(L))
    assert np.array_equal(np.stack([o.to_host() for o in outs]), exp)


@pytest.mark.parametrize("L,n_rows", [(17, 1 << 17), (18, (1 << 18) - 3), (18, 1 << 18), (20, (1 << 20) - 1)])
def test_combine_rows(vx, L, n_rows):
    rng = np.random.default_rng(n_rows)
    logs = [L, L - 3, L]
    spx, spy, fla = rnd(rng, 12), rnd(rng, 12), rnd(rng, 12)
    numers = [rnd(rng, 4, 1 << l) for l in logs]
    numers[0][:] = P - 1
    fla[:4] = [0, P - 1, 0, P - 1]
    dxs, dys = (d[:n_rows] for d in O.circle_domain_brev(L))
    exp = O.quotients_combine(spx, spy, fla, numers, logs, dxs, dys, L)
    assert np.array_equal(gpu_combine(vx, spx, spy, fla, numers, logs, dxs, dys, L, n_rows), exp)


@pytest.mark.parametrize("n_rows", [256, 768, (1 << 20) - 256, 1 << 20])
@pytest.mark.parametrize("n_batch", [3, 4, 9])
def test_numerator_rows(vx, n_rows, n_batch):
    rng = np.random.default_rng(n_rows + n_batch)
    cols = [rnd(rng, n_rows) for _ in range(4)]
    cols[1][:] = P - 1
    idx = rng.integers(0, 4, n_batch).astype(np.uint32)
    b, c = rnd(rng, 4 * n_batch), np.full(4 * n_batch, P - 1, np.uint32)
    assert np.array_equal(gpu_numerators(vx, cols, idx, b, c, n_rows), O.accumulate_numerators(cols, idx, b, c, n_rows))
