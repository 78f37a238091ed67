"""PoW search where most waves find a nonce at once: few bits, both sides of the line
from which a find is not looked up again, ranges that end inside a wave. Runs on the MI355X."""

import numpy as np
import pytest

import oracle_lib as O

pytestmark = pytest.mark.gpu
NONE = (1 << 64) - 1


@pytest.mark.parametrize("m31", [False, True])
@pytest.mark.parametrize("bits", [0, 1, 3, 6, 9, 10, 11, 13])
@pytest.mark.parametrize("offset,n", [(0, 1 << 20), ((1 << 32) - 100, 1 << 18), (12345, 63), (7, 129)])
def test_smallest_nonce(vx, bits, offset, n, m31):
    state = np.random.default_rng(100 * bits + m31).integers(0, 1 << 32, 8, dtype=np.uint64).astype(np.uint32)
    pre = O.pow_prefix(state, bits, m31)
    buf, result = vx.DeviceBuffer.from_host(pre), vx.DeviceBuffer.from_host(np.full(2, 0xFFFFFFFF, np.uint32))
    (vx.lib.cuda_grind_pow_m31_output if m31 else vx.lib.cuda_grind_pow)(buf.addr, result.addr, bits, offset, n)
    vx.synchronize()
    vx.check()
    assert int(result.to_host().view(np.uint64)[0]) == O.pow_search(pre, bits, m31, offset, n)
