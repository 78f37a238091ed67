"""Points of the twiddle-table kernels, on the CPU."""

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))


def test_every_point_read_is_held(tmp_path):
    exe = tmp_path / "table_points_test"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror",
                    os.path.join(HERE, "host", "table_points_test.cpp"), "-o", str(exe)], check=True)
    assert "table points: ok" in subprocess.run([str(exe)], check=True, capture_output=True, text=True).stdout
