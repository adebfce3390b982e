"""What the kernels' sources have to keep to, checked without a GPU."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "lfm3-1.7b-mi50_amd", "csrc")


@pytest.mark.parametrize("name", sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".h"))))
def test_barriers_are_fenced(name):
    """The bare barrier builtin orders no memory access for the compiler and waits for no LDS read in flight: a hand-over of
    LDS between waves goes through common.h's ring_barrier / lds_barrier (or __syncthreads)."""
    text = open(os.path.join(CSRC, name)).read()
    text = re.sub(r"//[^\n]*", "", text)
    allowed = 1 if name == "common.h" else 0
    assert text.count("__builtin_amdgcn_s_barrier") == allowed
    if allowed:
        body = text[text.index("ring_barrier()"):]
        assert re.search(r's_waitcnt\(vmcnt_imm\(N\) & ~0x0F00\);\s*asm volatile\("" ::: "memory"\);\s*'
                         r'__builtin_amdgcn_s_barrier\(\);\s*asm volatile\("" ::: "memory"\);', body)
