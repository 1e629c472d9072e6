"""Bookkeeping of kernels (indices into state arrays, counts, decisions) run on
the host: tests/native/kernel_logic.cpp compiles the kernel sources for the CPU
and runs one lane of them on arrays that end at an unreadable page."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CXX = shutil.which("amdclang++") or "/opt/rocm/bin/amdclang++"


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    if not os.path.exists(CXX):
        pytest.skip("no clang++ of ROCm")
    exe = str(tmp_path_factory.mktemp("native") / "kernel_logic")
    native = os.path.join(ROOT, "tests", "native")
    subprocess.run([CXX, "-x", "c++", "-std=c++17", "-O1", "-w", "-I", native, "-I",
                    os.path.join(ROOT, "xtb_amd", "csrc"), os.path.join(native, "kernel_logic.cpp"), "-o", exe],
                   check=True)
    return exe


@pytest.mark.parametrize("check", ["sub_products", "jacobi_unfinished", "sub_contraction", "sub_next"])
def test_kernel_logic(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True)
    assert r.returncode == 0, f"status {r.returncode}\n{r.stdout}{r.stderr}"
