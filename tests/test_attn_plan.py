"""The verify attention's key blocks (host-only queries). Lengths just past a rule's line keep the blocks
that measured faster there."""

from __future__ import annotations

import pytest

from dspark_rocm import _lib, ops


@pytest.mark.parametrize("hq,hk,m,d,keys,blocks", [
    (32, 8, 16, 128, 10007, 32),      # 320 blocks of 256 keys become one workgroup a CU
    (32, 8, 16, 128, 12288, 32),      # up to one and a half a CU
    (32, 8, 16, 128, 12289, 49),
    (32, 8, 16, 128, 8200, 33),       # 8 keys past 256 whole blocks: the last workgroups are short
    (32, 8, 1, 128, 10007, 40),       # one row tile
    (48, 12, 8, 128, 7000, 28),       # 12 heads in 22 blocks would be 264 workgroups
    (28, 7, 8, 128, 10007, 32),       # 7 in 32 are 224
    (24, 4, 8, 256, 6000, 47),        # head dim 256: 128 keys
    (24, 4, 16, 256, 5000, 20),       # six waves below 8192 keys: 256
    (24, 4, 16, 256, 10007, 53),
    (18, 3, 1, 256, 16500, 65),       # 86 blocks of 3 heads would be 258 workgroups
    (4, 1, 8, 256, 32768, 171),       # no more than 192 blocks of one head
])
def test_blocks(hq, hk, m, d, keys, blocks):
    assert ops.verify_attention_blocks(1, hq, hk, m, d, keys) == blocks


@pytest.mark.parametrize("hq,hk,d", [(32, 8, 128), (12, 2, 256), (24, 4, 256), (6, 1, 256), (48, 12, 128), (8, 2, 64)])
def test_workspace_stays_within_its_bound(hq, hk, d):
    """The bound an engine sizes its workspace by holds at every length, and holds the blocks' partials."""
    lib = _lib.load()
    for m in (1, 5, 16):
        bound = ops.attention_workspace_bound(1, hq, hk, d, m)
        rows = (hq // hk * m + 15) // 16 * 16
        for keys in [*range(60, 40000, 61), 8192, 8193, 16384, 16385, 32768, 1 << 20]:
            got = int(lib.dspark_verify_attention_workspace(1, hq, hk, m, d, keys))
            nb = ops.verify_attention_blocks(1, hq, hk, m, d, keys)
            assert got <= bound and (nb == 1 or got >= hk * nb * rows * (d + 2) * 4)
