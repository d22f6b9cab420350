"""Every workgroup barrier of the kernels waits for the wave's LDS stores: they use lds_barrier()
(wait and barrier in one statement) and never __syncthreads(), whose wait the compiler dropped
at the head of the GEMM tile loops."""
import glob
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lofloat_amd",
                    "csrc")


def _code(path):
    text = open(path).read()
    return re.sub(r"//[^\n]*", "", text)


@pytest.mark.parametrize("path", sorted(glob.glob(os.path.join(CSRC, "*.h*"))),
                         ids=os.path.basename)
def test_no_barrier_without_its_wait(path):
    code = _code(path)
    assert "__syncthreads" not in code and "__builtin_amdgcn_s_barrier" not in code
    for m in re.finditer(r"asm[^;]*s_barrier", code):
        assert re.search(r"s_waitcnt lgkmcnt\(0\)\\n\\ts_barrier", m.group(0)), m.group(0)
