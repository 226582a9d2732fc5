"""Waits written by hand in kernels whose asynchronous copies the compiler does not track.

A copy to LDS (global_load_lds) is read by other lanes after a barrier, so the wait before it is the source's
own.  A wait for all but a number of loads holds only while the compiler keeps that number of loads behind the
copies, which nothing checks: every wait is for all loads, or (LDS alone) for none.
"""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ziggy-llm_amd", "csrc")
KERNELS = [f for f in sorted(os.listdir(CSRC)) if "global_load_lds" in open(os.path.join(CSRC, f)).read()]


@pytest.mark.parametrize("name", KERNELS)
def test_waits_count_no_loads(name):
    waits = re.findall(r"s_waitcnt\((\w+)\)", open(os.path.join(CSRC, name)).read())
    assert waits
    for w in waits:
        imm = int(w, 0)
        assert (imm & 0xF) | (imm >> 14 & 3) << 4 in (0, 63), f"{name}: partial vmcnt at {w}"  # bits 3:0 and 15:14
