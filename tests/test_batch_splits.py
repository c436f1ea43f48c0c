"""Split counts of a uniform batch: whole rounds of work-groups, never a second round
for a few of them."""

from __future__ import annotations

import pytest

from breezetoken_amd import _lib


@pytest.mark.parametrize("batch,heads,kv,length,expect", [
    (24, 8, 2, 3000, 5),     # 240 work-groups; 6 would be 288
    (48, 8, 2, 3000, 5),     # 480 in two rounds; 2 leave a quarter of the CUs idle
    (64, 8, 2, 3000, 4),
    (24, 32, 8, 3000, 4),    # 768 in three rounds
    (64, 8, 2, 400, 2),      # short: one round
    (1, 8, 2, 1, 1),
    (1, 8, 2, 65, 1),        # one split needs no combine
    (1, 8, 2, 1000, 32),     # at most a split per 32 tokens
    (5000, 8, 2, 8192, 1),
    (0, 0, 0, 0, 1),         # out-of-range sizes are clamped, as bt_decode_pick_splits does
])
def test_pick_splits_batch(batch, heads, kv, length, expect):
    assert _lib.lib().bt_decode_pick_splits_batch(batch, heads, kv, length, 256) == expect
