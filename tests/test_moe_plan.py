"""The routed-expert block's choice between its small-bucket kernels and the one for prompt chunks
(host-only queries): sizes where each measured faster."""

from __future__ import annotations

import pytest

from dspark_rocm import _lib, ops


@pytest.mark.parametrize("m,e,k,h,i,bits,rows", [
    (96, 128, 8, 2048, 768, 4, True), (95, 128, 8, 2048, 768, 4, False),      # six rows an expert, top 8
    (500, 128, 8, 2048, 768, 8, True),
    (64, 8, 2, 2048, 768, 4, False), (144, 8, 2, 2048, 768, 4, True),         # few experts, few pairs
    (96, 8, 2, 2048, 768, 8, True),
    (32, 8, 2, 1024, 384, 4, False), (100, 8, 4, 1024, 384, 8, False),
    (48, 64, 8, 512, 256, 4, False), (64, 64, 8, 512, 256, 4, True),          # small experts
    (24, 16, 2, 4096, 1536, 4, True), (17, 4, 1, 4096, 1536, 8, True), (17, 4, 1, 4096, 1536, 4, False),
    (24, 16, 1, 2560, 384, 8, False), (240, 16, 1, 2560, 384, 8, True),
    (16, 4, 4, 4096, 1536, 8, False),                                         # a verify block never
])
def test_prompt_chunks_take_the_faster_kernels(m, e, k, h, i, bits, rows):
    plan = ops.moe_packed_plan(m, h, i, e, k, bits)
    assert [plan[s] == "row tiles" for s in ("gate_up", "down")] == [rows, rows]


def test_workspace_covers_both_widths():
    """One query for both widths, whichever kernels each takes: the larger need."""
    lib = _lib.load()
    m, e, k, h, i = 96, 8, 2, 2048, 768                     # 8 bits by row tiles, 4 bits not
    sums = 2 * 3 * (m * 32 + m * k * 32)                    # three bf16 pieces of 32 group sums a row
    pairs = 2 * m * k * (h + i)                             # h and y
    assert int(lib.dspark_moe_workspace(m, h, i, e, k)) >= sums + pairs
