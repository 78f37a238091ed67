"""accumulate_numerators on both sides of its rules: rows from which a thread takes
four and eight, plain or global loads, columns past whole groups of four, unaligned
columns and outputs, against the oracle on rows of every part. Runs on the MI355X."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


ROWS = [1, 255, 256, 768, (1 << 19) - 256, 1 << 19, (1 << 20) - 256, 1 << 20, 3 << 19, (3 << 19) + 256]
CASES = [(n, r, 0, 0) for n in (1, 2, 3, 4, 7, 8, 9, 10, 11) for r in ROWS]
CASES += [(n, r, cs, 1 - cs) for n in (3, 8) for r in ROWS for cs in (0, 1)]


@pytest.mark.parametrize("n_cols,n_rows,col_shift,out_shift", CASES)
def test_rules(vx, n_cols, n_rows, col_shift, out_shift):
    rng = np.random.default_rng(n_rows + 16 * n_cols)
    draw = lambda n: rng.integers(0, P, n, dtype=np.uint64).astype(np.uint32)  # noqa: E731
    cols, b, c = [draw(n_rows) for _ in range(n_cols)], draw(4 * n_cols), draw(4 * n_cols)
    cols[0][-1] = P - 1
    c[:4] = P - 1
    idx = np.arange(n_cols, dtype=np.uint32)[::-1].copy()
    pad = np.zeros(col_shift, np.uint32)
    bufs = [vx.DeviceBuffer.from_host(np.concatenate([pad, x])) for x in cols]
    outs = [vx.DeviceBuffer(n_rows + out_shift) for _ in range(4)]
    dev = [vx.DeviceBuffer.from_host(x) for x in
           (np.array([x.addr + 4 * col_shift for x in bufs], np.uint64).view(np.uint32), idx, b, c)]
    vx.lib.cuda_accumulate_numerators(*[d.addr for d in dev], n_cols, n_rows, *[o.addr + 4 * out_shift for o in outs])
    vx.synchronize()
    vx.check()
    # the first and last rows of the batch and of a thread's, a wave's and a workgroup's share
    at = sorted({r for e in (0, 1, 4, 64, 256, 512, 1024, 2048, n_rows // 2, n_rows - 512, n_rows)
                 for r in (e - 1, e, e + 3) if 0 <= r < n_rows})
    want = O.accumulate_numerators([x[at] for x in cols], idx, b, c, len(at))
    got = np.stack([o.to_host()[out_shift:][at] for o in outs])
    assert np.array_equal(got, np.asarray(want).reshape(4, len(at)))
