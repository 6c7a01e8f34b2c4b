"""Division by a launch constant (cpml_constdiv.h) against the IEEE division,
on the CPU: bit for bit over a spread of significands in float (every binade
kind: smallest allowed, middle, largest; signed zeros) and random doubles."""
import shutil
import subprocess
from pathlib import Path

import pytest

SRC = Path(__file__).resolve().parent / "native" / "const_div_check.cpp"


def test_const_div_equals_division(tmp_path):
    # the compiler family of the device code (g++ folds -fma(a, b, -c) into
    # c - a b, which loses the sign of a zero)
    cxx = shutil.which("amdclang++") or shutil.which("clang++") or "/opt/rocm/llvm/bin/clang++"
    if not Path(cxx).exists():
        pytest.skip("no clang++")
    exe = tmp_path / "const_div_check"
    subprocess.run([cxx, "-O2", "-mfma", "-std=c++17", "-ffp-contract=off", str(SRC), "-o",
                    str(exe)], check=True)
    r = subprocess.run([str(exe), "61"], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout
    assert int(r.stdout.split()[0]) > 10_000_000
