"""Transforms of every small size (a tile of fewer groups than its workgroup has
threads) and of the two-pass sizes without a plan, native and stwo basis, both
directions, aligned and not, against the oracle. Runs on the MI355X."""

import ctypes as C

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


@pytest.mark.parametrize("k", list(range(1, 15)) + [20, 21, 22, 23])
def test_sizes(vx, k):
    vx.lib.vx_ntt_plan_reset()
    n = 1 << k
    x = np.random.default_rng(k).integers(0, P, n + 1, dtype=np.uint64).astype(np.uint32)
    line, circle, iline, icircle, offs, sizes = O.ntt_twiddles(1, k)
    tabs = [vx.DeviceBuffer.from_host(t) for t in (line, circle, iline, icircle)]
    ho, hs = ((C.c_uint32 * max(1, k - 1))(*[int(v) for v in a[: k - 1]]) for a in (offs, sizes))
    for shift in (0, 1):
        buf = vx.DeviceBuffer.from_host(x)
        at, part = buf.addr + 4 * shift, x[shift: shift + n]
        exp = part.copy()
        O.lib().orc_ntt_evaluate(exp.ctypes.data, line.ctypes.data, circle.ctypes.data, k)
        vx.lib.cuda_circle_ntt_evaluate(at, tabs[0].addr, tabs[1].addr, ho, hs, k - 1, n)
        vx.check("evaluate")
        assert np.array_equal(buf.to_host()[shift: shift + n], exp)
        vx.lib.cuda_circle_ntt_interpolate(at, tabs[2].addr, tabs[3].addr, ho, hs, k - 1, n)
        vx.check("interpolate")
        assert np.array_equal(buf.to_host(), x)  # the neighbouring word too
        if k < 2:
            continue
        sf, si = O.stwo_twiddles(k)
        dsf, dsi = vx.DeviceBuffer.from_host(sf), vx.DeviceBuffer.from_host(si)
        exp = part.copy()
        O.lib().orc_stwo_ntt_evaluate(exp.ctypes.data, sf.ctypes.data, k)
        vx.lib.cuda_stwo_ntt_evaluate(at, dsf.addr, n)
        vx.check("stwo evaluate")
        assert np.array_equal(buf.to_host()[shift: shift + n], exp)
        vx.lib.cuda_stwo_ntt_interpolate(at, dsi.addr, n)
        vx.check("stwo interpolate")
        assert np.array_equal(buf.to_host(), x)
