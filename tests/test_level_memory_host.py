"""The level driver's host code where device memory runs out, without a GPU:
tests/level_memory_host.cpp links the built library and stands in for the HIP
runtime's memory calls (tests/host_runtime.h; kernels do not run)."""
import os
import shutil
import subprocess

import pytest

from camr_amd import _lib

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.mark.skipif(not shutil.which("g++"), reason="g++ not available")
def test_memory_that_buys_speed_is_given_up_first(tmp_path):
    exe = tmp_path / "level_memory_host"
    libdir = os.path.dirname(_lib.LIB_PATH)
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wno-unused-result", "-o", str(exe),
                    os.path.join(ROOT, "tests", "level_memory_host.cpp"),
                    "-I", os.path.join(ROOT, "include"), "-I", "/opt/rocm/include",
                    "-L", libdir, "-lcamr_hydro", "-Wl,-rpath," + libdir,
                    "-L", "/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib", "-lamdhip64"],
                   check=True, capture_output=True, timeout=300)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=300)
    print(out.stdout, out.stderr)
    assert out.returncode == 0 and "LEVEL MEMORY OK" in out.stdout, out.stdout[-3000:]
