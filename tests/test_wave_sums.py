"""The sums over a wave that wrap: in the compiler's intermediate code they are additions that may, so that nothing can be concluded
from their not wrapping."""
import os
import re
import shutil
import subprocess

import pytest

import lbtree

_CSRC = os.path.join(os.path.dirname(os.path.dirname(lbtree.__file__)), "csrc")
_KERNEL = """#include "lbt_device.h"
extern "C" __global__ void summed(const uint32_t* v, uint32_t* out) { out[threadIdx.x] = lbt::wave_inclusive_sum32(v[threadIdx.x]); }
"""


@pytest.mark.skipif(shutil.which("hipcc") is None, reason="needs hipcc")
def test_sums_of_32_bits_may_wrap(tmp_path):
    source, code = tmp_path / "summed.hip", tmp_path / "summed.ll"
    source.write_text(_KERNEL)
    subprocess.run(["hipcc", "-O1", "-std=c++17", "--offload-arch=gfx950", "--cuda-device-only", "-S", "-emit-llvm", "-I" + _CSRC,
                    str(source), "-o", str(code)], check=True, capture_output=True)
    body = re.search(r"define [^\n]*@summed\(.*?^}", code.read_text(), re.S | re.M).group(0)
    additions = re.findall(r"= (add[^\n]*) i32 ", body)
    assert additions == ["add"] * 6
