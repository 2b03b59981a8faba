"""Quotients that the kernels form without a division, compiled for the CPU from the library's own header and compared with the
division: that of every draw by its range, and those from an approximate reciprocal on operands as the gains have them."""
import os
import shutil
import subprocess

import pytest

import lbtree

_CSRC = os.path.join(os.path.dirname(os.path.dirname(lbtree.__file__)), "csrc")


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_quotients_are_those_of_the_division(tmp_path):
    source, program = os.path.join(os.path.dirname(os.path.abspath(__file__)), "quotients.cpp"), str(tmp_path / "quotients")
    subprocess.run(["hipcc", "-x", "hip", "--offload-host-only", "-O2", "-std=c++17", "-march=x86-64-v3", "-ffp-contract=off", "-pthread",
                    "-I" + _CSRC, source, "-o", program], check=True, capture_output=True)
    out = subprocess.run([program], check=True, capture_output=True, text=True).stdout
    assert out.split() == ["0", "0"]
