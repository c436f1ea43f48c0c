"""Split counts of a uniform batch by head dimension: the counts asserted are the measured
faster ones (us beside them, this count against the one it is not)."""

from __future__ import annotations

import pytest

from breezetoken_amd import _lib


@pytest.mark.parametrize("batch,heads,kv,dim,length,expect", [
    (33, 32, 8, 128, 300, 1),      # 8.8; 2 splits 14.5
    (33, 32, 8, 64, 300, 1),       # 5.8; 2 splits 9.8
    (128, 16, 2, 256, 2000, 1),    # 70.7, a work-group per CU; 2 splits 86.2
    (128, 16, 2, 128, 3000, 1),    # 51.6; 3 splits 60.1
    (64, 8, 2, 256, 300, 1),       # 10.9; 2 splits 16.8
    (1, 8, 2, 256, 20000, 128),    # 12.1; 127 splits 12.8
    (4, 6, 2, 64, 8000, 32),       # 7.7; 31 splits 8.1
    (2, 32, 8, 128, 1000, 16),     # 7.0; 15 splits 7.3
    (24, 8, 2, 256, 3000, 5),      # 31.3; 6 splits, 288 work-groups, 43.2
    (24, 32, 8, 128, 3000, 4),     # 43.1 in three rounds; 2 splits 48.7
    (33, 32, 8, 128, 3000, 4),     # 60.3; one split, 264 work-groups, 75.1
    (64, 8, 2, 256, 3000, 4),      # 59.8; 2 splits 62.9
    (1, 8, 2, 256, 1, 1),
    (1, 8, 2, 256, 65, 1),
    (0, 0, 0, 0, 0, 1),            # out-of-range sizes are clamped
    (5000, 8, 2, 256, 8192, 1),
])
def test_pick_splits_uniform(batch, heads, kv, dim, length, expect):
    assert _lib.lib().bt_decode_pick_splits_uniform(batch, heads, kv, dim, length, 256) == expect


@pytest.mark.parametrize("dim", [64, 128, 256])
@pytest.mark.parametrize("pairs", [1, 2, 3, 7, 24, 64, 100, 255, 256, 257, 300, 1000])
def test_counts_stay_in_range(pairs, dim):
    for length in (1, 31, 32, 33, 500, 4000, 100000, 2**31 - 1):
        ns = _lib.lib().bt_decode_pick_splits_uniform(pairs, 4, 1, dim, length, 256)
        assert 1 <= ns <= min(-(-length // 32), max(1, 5 * 256 // pairs))
