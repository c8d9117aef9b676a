"""A bare s_barrier orders nothing by itself.  Where tiles go through a ring in LDS, the stage that is asked for behind the barrier is the
one that was read in front of it, so each wave has to have waited for its own reads as well as for its loads."""
import os
import re

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "turboquant.cpp_amd", "csrc")


@pytest.mark.parametrize("name", ["gemm_f32.hip", "gemm_mfma.hip"])
def test_rings_wait_for_their_reads(name):
    with open(os.path.join(CSRC, name)) as f:
        parts = f.read().split("__builtin_amdgcn_s_barrier()")
    assert len(parts) > 1
    for before in parts[:-1]:
        waits = re.findall(r"__builtin_amdgcn_s_waitcnt\((0x[0-9A-Fa-f]{4})", before)[-2:]      # with loads left, and at the end
        # lgkmcnt stands in bits 11..8: 0 asks for the reads of LDS
        assert len(waits) == 2 and all(int(w, 16) >> 8 & 15 == 0 for w in waits), (name, waits)
