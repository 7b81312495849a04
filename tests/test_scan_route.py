"""Which scans run with time across the lanes (csrc/scan_lanes.hip's plan) and which on the general
kernel: host-only, on either side of the rule's lines.  Where a call goes was measured; these
cases keep it there."""

from __future__ import annotations

import pytest
import torch

from helpers import scan_route

F32, F16, BF16 = torch.float32, torch.float16, torch.bfloat16

# (layout, dtype, batch, dim, dstate, seqlen, waves per channel, segments)
LANES = [
    ("bdl", F32, 1, 16, 16, 4096, 4, 8), ("bdl", F32, 1, 16, 16, 32768, 4, 64), ("bdl", BF16, 3, 1000, 16, 3001, 2, 1),
    ("bld", F16, 1, 1536, 16, 2048, 1, 1), ("bld", BF16, 3, 2048, 16, 777, 1, 1), ("bld", F32, 2, 1024, 16, 1021, 2, 1),
    ("bdl", F16, 1, 8, 16, 8, 4, 1), ("bdl", F16, 1, 1536, 16, 512, 4, 1), ("bdl", F16, 1, 1024, 16, 64, 4, 1),
    ("bdl", F16, 1, 4096, 16, 2048, 1, 1), ("bdl", F16, 1, 2560, 16, 896, 2, 1), ("bdl", F16, 1, 2048, 16, 1152, 2, 1),
    ("bdl", F16, 1, 3072, 16, 4096, 2, 1), ("bdl", F32, 1, 1024, 16, 16384, 4, 1), ("bdl", F16, 1, 256, 16, 2048, 4, 4),
    ("bdl", F16, 1, 128, 16, 16384, 1, 32), ("bdl", F16, 1, 512, 4, 2048, 2, 4), ("bdl", F16, 1, 5120, 4, 4608, 1, 1),
    ("bld", F16, 1, 1024, 16, 1024, 2, 1), ("bld", F32, 4, 1024, 16, 16384, 2, 1), ("bld", F16, 1, 256, 16, 2048, 2, 4),
    ("bdl", F16, 1, 16, 32, 65536, 4, 1), ("bdl", F16, 1, 16384, 24, 512, 1, 1), ("bld", F16, 1, 12288, 32, 512, 1, 1),
]
GENERAL = [
    ("bdl", F16, 1, 16, 16, 7), ("bdl", F16, 8, 1536, 16, 8192), ("bdl", F16, 4, 5120, 16, 32768),
    ("bdl", F16, 1, 2560, 16, 768), ("bdl", F16, 1, 2560, 16, 1152), ("bdl", F16, 1, 2560, 16, 2304),
    ("bdl", F16, 1, 2560, 16, 8192), ("bdl", F16, 1, 1280, 16, 1152), ("bdl", F16, 1, 5120, 16, 1152),
    ("bdl", F16, 2, 1536, 16, 16384), ("bdl", F16, 1, 512, 16, 1280), ("bdl", F16, 1, 256, 16, 4608),
    ("bdl", F32, 1, 256, 16, 4608), ("bdl", F32, 1, 1536, 8, 12288), ("bdl", F32, 1, 2560, 16, 640),
    ("bld", F16, 1, 2560, 16, 768), ("bld", F32, 1, 1280, 16, 4096), ("bld", F32, 4, 1024, 8, 32768),
    ("bld", F16, 2, 1536, 16, 16384), ("bld", F16, 1, 1024, 16, 2048), ("bld", F16, 1, 16, 12, 4096),
    ("bld", F16, 1, 16384, 32, 1024), ("bdl", F16, 1, 16384, 64, 1024), ("bdl", F16, 1, 1024, 16, 32768),
]


@pytest.mark.parametrize("layout,dtype,batch,dim,dstate,seqlen,waves,segments", LANES, ids=str)
def test_lanes(layout, dtype, batch, dim, dstate, seqlen, waves, segments):
    assert scan_route(layout, dtype, batch, dim, dstate, seqlen) == (waves, segments)
    # other types of B and C: scan_kernel's packed copies
    assert scan_route(layout, dtype, batch, dim, dstate, seqlen, bc_dtype=F32 if dtype != F32 else F16)[0] == 0


@pytest.mark.parametrize("layout,dtype,batch,dim,dstate,seqlen", GENERAL, ids=str)
def test_general(layout, dtype, batch, dim, dstate, seqlen):
    assert scan_route(layout, dtype, batch, dim, dstate, seqlen)[0] == 0


def test_no_room_for_summaries():
    """A workspace without segment summaries (the allocation-free entry point's, for some batches): one
    pass over all chunks."""
    assert scan_route("bdl", F16, 32, 2, 16, 4096) == (4, 8)
    assert scan_route("bdl", F16, 32, 2, 16, 4096, workspace_bytes=1 << 20) == (4, 1)
