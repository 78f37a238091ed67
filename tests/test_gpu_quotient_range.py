"""The Fibonacci quotient at the largest sizes its 32-bit arguments allow. Runs on the MI355X."""

import ctypes as C

import pytest

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


# The last four words of a trace of 2^32 - 1 (and fewer) words lie past every whole
# group of four, at indices whose successor group begins past 2^32. All four outputs
# share one buffer and one factor, so the call takes 16 GiB beside the 16 GiB trace.
@pytest.mark.parametrize("n", [(1 << 32) - 1, (1 << 32) - 3, (1 << 32) - 4])
def test_last_words(vx, n):
    trace, out = vx.DeviceBuffer(n), vx.DeviceBuffer(n)
    vx.lib.vx_memset(trace.addr, 0x11, 4 * n)
    vx.lib.vx_memset(out.addr, 0xFF, 4 * n)
    alpha = 12345
    vx.lib.cuda_fibonacci_quotient(trace.addr, *[out.addr] * 4, (C.c_uint32 * 4)(*[alpha] * 4), n)
    vx.synchronize()
    vx.check("cuda_fibonacci_quotient")
    want = (P - 0x11111111) * alpha % P  # t - (t + t)
    for at in (0, n // 2, n - 8):
        assert (vx.device_copy_words(out.addr + 4 * at, 8) == want).all(), at
    trace.free()
    out.free()
