"""Rules of cudart_amd/csrc/kernels/launch_shape.hpp, compiled for the CPU
(tests/host_launch_shape.cpp): the spill columns asked for are enough for every thread of every
launch of a call, whatever the image, the sample count and the launch size, an allocation
that fails leaves the area that was there, a launch of any number of resident waves hands out
every batch of its queue, and idle memory is bounded by the device's and by what is free."""
import subprocess
from pathlib import Path

ROOT = Path(__file__).resolve().parent.parent


def test_rules_hold_over_the_accepted_sizes(tmp_path):
    exe = tmp_path / "shapes"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Wextra", "-Werror", "-fsanitize=undefined",
                    "-fno-sanitize-recover=all", f"-I{ROOT / 'cudart_amd' / 'csrc' / 'kernels'}",
                    str(ROOT / "tests" / "host_launch_shape.cpp"), "-o", str(exe)], check=True, timeout=120)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=120)
    assert out.returncode == 0, out.stdout + out.stderr
