"""Fold-twiddle sources of every domain whose index has fewer bits than a workgroup's
run numbers, and of the first ones with more, against the points themselves. Runs on
the MI355X."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
P = (1 << 31) - 1


def mul(a, b):
    return (a[0] * b[0] - a[1] * b[1]) % P, (a[0] * b[1] + a[1] * b[0]) % P


@pytest.mark.parametrize("use_y", [0, 1])
@pytest.mark.parametrize("log_n", range(1, 15))
def test_sources(vx, log_n, use_y):
    n, half = 1 << log_n, 1 << (log_n - 1)
    step = (2, 1268011823)  # of order 2^31
    for _ in range(31 - log_n):
        step = mul(step, step)
    initial = (717131204 % P, 5)  # any point: the sources are products, on the circle or not
    out = vx.DeviceBuffer.from_host(np.full(half + 1, 0xFFFFFFFF, np.uint32))
    vx.lib.cuda_compute_fold_twiddle_sources(*initial, *step, out.addr, n, log_n, use_y)
    vx.synchronize()
    vx.check()
    p, want = initial, np.zeros(half, np.uint32)
    for j in range(half):  # word i holds exponent j = bit reversal of i in log_n - 1 bits
        i = int(format(j, "0%db" % (log_n - 1))[::-1], 2) if log_n > 1 else 0
        want[i] = p[use_y]
        p = mul(p, step)
    got = out.to_host()
    assert np.array_equal(got[:-1], want) and got[-1] == 0xFFFFFFFF
