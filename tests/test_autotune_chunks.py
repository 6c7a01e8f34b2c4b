"""The autotuner's chunk depths hold the default of the shape that it times, so it
never ends with a slower one (CPU, through the library's own header)."""
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "native" / "autotune_chunks_check.cpp"
CXX = Path("/opt/rocm/llvm/bin/clang++")


def test_autotuner_times_the_default(tmp_path):
    if not CXX.exists():
        pytest.skip("no clang++")
    exe = tmp_path / "autotune_chunks_check"
    subprocess.run([str(CXX), "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(SRC), "-o", str(exe)], check=True)
    r = subprocess.run([str(exe)], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
