"""Launch shapes and row walks at row counts that no test can allocate (CPU):
tests/cxx/launch_shapes_check.cpp runs the host's shape rules and the kernels'
own row walk (csrc/launch_shapes.hpp) up to the largest counts that the calls
admit, under the undefined-behaviour sanitizer."""
import os
import subprocess

from munet_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def test_row_walks_stay_in_range(tmp_path):
    exe = str(tmp_path / "check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-D__host__=",
                        "-D__device__=", "-D__forceinline__=inline", "-I", build.CSRC,
                        os.path.join(ROOT, "tests", "cxx", "launch_shapes_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]
