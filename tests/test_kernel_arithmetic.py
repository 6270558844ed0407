"""Arithmetic of the kernels that can be checked whole without a GPU: the addresses their requests ask for, and the
exponential and the division in fewer instructions."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "llama.cu_amd", "csrc")
CXX = os.path.join(ROOT, "tests", "cxx")


@pytest.fixture(scope="module")
def operand_range(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("range") / "operand_range")
    subprocess.run(["g++", "-O2", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, os.path.join(CXX, "operand_range.cpp"), "-o", exe], check=True)
    return exe


def test_requests_stay_in_their_operands(operand_range):
    res = subprocess.run([operand_range], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout


def test_a_scalar_offset_without_a_length_would_be_found(operand_range):
    res = subprocess.run([operand_range, "offset"], capture_output=True, text=True)
    assert res.returncode == 1 and " 0 reach" not in res.stdout, res.stdout


def test_short_exponential_and_division(tmp_path):
    """exp_ieee_nonpositive has exp_ieee's bits, and divide_by the quotient's where the kernels use it."""
    exe = str(tmp_path / "kernel_arithmetic")
    subprocess.run(["hipcc", "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-ffp-contract=off", "-mfma", "-mf16c", "-I", CSRC,
                    "-I", os.path.join(ROOT, "include"), os.path.join(CXX, "kernel_arithmetic.hip"), "-o", exe], check=True)
    res = subprocess.run([exe], capture_output=True, text=True)
    assert res.returncode == 0, res.stdout
