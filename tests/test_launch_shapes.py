"""Launch shapes, row walks and tile choices at sizes that no test can allocate
or time (CPU): tests/cxx/*_check.cpp run the host's rules and the kernels' own
row walk (csrc/launch_shapes.hpp, csrc/gemm_tiles.hpp) up to the largest counts
that the calls admit, under the undefined-behaviour sanitizer."""
import os
import subprocess

import pytest

from munet_amd import build

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.parametrize("name", ["launch_shapes", "gemm_tiles"])
def test_launch_rules(name, tmp_path):
    exe = str(tmp_path / "check")
    r = subprocess.run(["g++", "-std=c++17", "-O1", "-fsanitize=undefined", "-fno-sanitize-recover=all", "-D__host__=",
                        "-D__device__=", "-D__forceinline__=inline", "-I", build.CSRC,
                        os.path.join(ROOT, "tests", "cxx", name + "_check.cpp"), "-o", exe],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([exe], capture_output=True, text=True, timeout=120)
    assert r.returncode == 0 and r.stdout == "ok\n", r.stdout + r.stderr[-2000:]
