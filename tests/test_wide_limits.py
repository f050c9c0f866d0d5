"""Sizes the many-row product refuses on the host: a launch has fewer than 2^32 threads, 8 of them for
each group sum of x (rows times groups of 64, the groups padded to a multiple of 32)."""

from __future__ import annotations

import pytest

from dspark_rocm import _lib


@pytest.mark.parametrize("m,k,ok", [(1 << 23, 64, True), ((1 << 23) + 1, 64, False), (1 << 24, 64, False),
                                    (1 << 23, 2048, True), (1 << 23, 2112, False), (1 << 22, 4096, True),
                                    ((1 << 22) + 1, 4096, False), (1 << 12, 1 << 22, True)])
def test_group_sums_fit_one_launch(m, k, ok):
    assert (int(_lib.load().dspark_qmm_wide_workspace(m, k, 128, 8, 64)) > 0) == ok
