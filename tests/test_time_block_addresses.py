"""Items and addresses of the marches without a hardware range check -- time-blocked
2D, batch and 3D (cpml_tb_geom.h) and the ADE-RK4 pairs (cpml_ade8_split.h) -- on the
CPU, through the code that the kernels compile, over random grids, slabs, strip
widths and chunk depths: what is loaded and stored lies inside its array, and
each point of the grid is stored once.  The memory variables have no ghost points: with the
fields' clamp (to the ghost column nx) narrow strips read past their rows, and
the audit has to say so."""
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "native" / "address_audit.cpp"
CXX = Path("/opt/rocm/llvm/bin/clang++")


@pytest.fixture(scope="module")
def audit(tmp_path_factory):
    if not CXX.exists():
        pytest.skip("no clang++")
    exe = tmp_path_factory.mktemp("audit") / "address_audit"
    subprocess.run([str(CXX), "-O2", "-std=c++17", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    str(SRC), "-o", str(exe)], check=True)
    return lambda *a: subprocess.run([str(exe), *a], capture_output=True, text=True)


def test_addresses_in_bounds(audit):
    r = audit("200")
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 1_000_000_000


def test_audit_finds_ghost_columns_of_memory_variables(audit):
    r = audit("20", "ghost")
    assert r.returncode == 1 and "y memory" in r.stdout and "z memory" in r.stdout
