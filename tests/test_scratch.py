"""The pool of device temporaries that contexts keep between calls (mpqc_amd/csrc/scratch.hpp), on a
made-up device: its bound over all contexts, who gets a block, and when blocks go back."""
import pathlib
import shutil
import subprocess

import pytest

HERE = pathlib.Path(__file__).resolve().parent


def test_scratch_pool(tmp_path):
    gxx = shutil.which("g++")
    rocm = pathlib.Path("/opt/rocm/include/hip/hip_runtime_api.h")
    if gxx is None or not rocm.exists():
        pytest.skip("g++ or the HIP headers are not available")
    exe = tmp_path / "scratch_check"
    subprocess.run([gxx, "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I", str(rocm.parents[1]),
                    str(HERE / "scratch_check.cpp"), "-o", str(exe), "-pthread"], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=60)
    print(out.stdout)
    assert out.returncode == 0, out.stdout + out.stderr
