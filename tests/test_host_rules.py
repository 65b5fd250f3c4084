"""Host-side rules of the native library, compiled without a GPU and run here: each program in
tests/host/ includes the library's own sources and returns 0, or prints what it found."""
import os
import shutil
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(os.path.dirname(HERE), "beast.jl_amd", "csrc")


@pytest.mark.skipif(shutil.which("g++") is None, reason="needs a host compiler")
@pytest.mark.parametrize("name", ["tournament_sets", "panel_positions", "panel_gate", "pool_sizes", "pool_pressure", "tile_groups", "pair_groups", "results"])
def test_host_program(name, tmp_path):
    exe = str(tmp_path / name)
    # the platform macro: HIP's headers need it from a compiler other than hipcc
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-pthread", "-D_GLIBCXX_ASSERTIONS", "-D__HIP_PLATFORM_AMD__",
                    "-I", CSRC, "-I", "/opt/rocm/include", os.path.join(HERE, "host", name + ".cpp"), "-o", exe], check=True)
    r = subprocess.run([exe], capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stdout + r.stderr
