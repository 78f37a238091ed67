"""Fibonacci traces longer than a domain: steps and grid on the CPU, words on the MI355X."""

import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
P = (1 << 31) - 1


def test_steps_and_grid(tmp_path):
    exe = tmp_path / "trace_plan_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(HERE, "host", "trace_plan_test.cpp"), "-o", str(exe)], check=True)
    assert "trace plan: ok" in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout


def fib(k):
    """(F(k), F(k + 1)) mod p by doubling."""
    if k == 0:
        return 0, 1
    x, y = fib(k // 2)
    u, v = x * (2 * y - x) % P, (x * x + y * y) % P
    return (v, (u + v) % P) if k & 1 else (u, v)


def trace_word(a, b, i):
    if i == 0:
        return a
    f, g = fib(i - 1)  # F(i - 1), F(i)
    return (f * a + g * b) % P


@pytest.mark.gpu
@pytest.mark.parametrize("log_n", [0, 3, 12, 33])  # 2^33 words are 32 GiB
def test_words(vx, log_n):
    a, b, n = 123456789, 987654321, 1 << log_n
    trace = vx.fibonacci_trace_device(a, b, log_n)
    for i in sorted(i for i in {0, 1, n // 3, n // 2 - 1, n // 2, n - 17, n - 1} if 0 <= i < n):
        assert int(vx.device_copy_words(trace.addr + 4 * i, 1)[0]) == trace_word(a, b, i), i
    if n >= 8:
        tail = vx.device_copy_words(trace.addr + 4 * (n - 8), 8).astype(np.uint64)
        assert np.array_equal(tail[2:], (tail[:-2] + tail[1:-1]) % P)
    trace.free()
