"""Bytes that the benchmark reports for the ADE-RK4 step: the box that takes two
stages per pass is the kernels' (through their own header, on the CPU), and a step
moves 41 words per point inside it and 92 outside."""
import subprocess
from pathlib import Path
from types import SimpleNamespace

import pytest

from seismic_cpml_amd import workloads

SRC = Path(__file__).resolve().parent / "native" / "ade8_box.cpp"
CXX = Path("/opt/rocm/llvm/bin/clang++")


def test_box_and_bytes(tmp_path):
    if not CXX.exists():
        pytest.skip("no clang++")
    exe = tmp_path / "ade8_box"
    subprocess.run([str(CXX), "-O1", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(SRC), "-o", str(exe)], check=True)
    for nx, ny, npml, prec in [(4096, 4096, 20, 4), (4096, 4096, 20, 8), (1200, 1000, 10, 4),
                               (1200, 1000, 10, 8), (500, 600, 20, 4), (3000, 90, 0, 8),
                               (5001, 777, 3, 4)]:
        r = subprocess.run([str(exe), *map(str, (nx, ny, npml, prec))], capture_output=True,
                           text=True, check=True)
        box = tuple(map(int, r.stdout.split()))
        assert workloads.ade8_pair_box(nx, ny, npml, prec) == box
        inside = (box[1] - box[0]) * (box[3] - box[2])
        w = SimpleNamespace(nx=nx, ny=ny, npml=npml, prec=prec, cells=nx * ny)
        assert workloads.ade8_own_bytes(w) == prec * (41 * inside + 92 * (nx * ny - inside))
