"""Which prefill kernel a call takes, by the library's estimate of both (bt_prefill_plan;
256 CUs where no GPU is present).  The choices asserted are the measured faster ones."""

from __future__ import annotations

import ctypes

import pytest

from breezetoken_amd import _lib

ALL = 1 << 40  # room for any partials


def prefill_plan(steps, heads, kv, dim, q_f32, room=ALL, q_offset=0):
    out = (ctypes.c_int32 * 5)()
    _lib.check("bt_prefill_plan", _lib.lib().bt_prefill_plan(
        steps, q_offset, heads, kv, dim, _lib.BT_DTYPE_F32 if q_f32 else _lib.BT_DTYPE_BF16, room,
        ctypes.addressof(out)))
    return dict(zip(("pair", "chunk", "chunks", "order", "parts"), out))


# us, pair kernel against two waves per SIMD
@pytest.mark.parametrize("steps,heads,kv,dim,q_f32,pair", [
    (256, 8, 2, 256, True, False),     # 24.1 / 23.2
    (256, 16, 2, 128, True, False),    # 16.6 / 15.5
    (1024, 8, 2, 256, True, True),     # 41.0 / 50.9
    (1024, 8, 2, 256, False, False),   # 52.6 / 40.7
    (2048, 8, 2, 256, False, False),   # 80.3 / 68.7
    (3001, 8, 2, 256, False, False),   # 104 / 95
    (3001, 8, 2, 256, True, True),     # 82 / 120
    (1500, 16, 2, 256, False, False),  # 66.7 / 55.9
    (2048, 4, 4, 256, False, False),   # 83.5 / 71.1
])
def test_calls_without_partials_take_the_faster_kernel(steps, heads, kv, dim, q_f32, pair):
    """Grids that leave CUs idle, where the two-wave kernel's blocks are faster than under load."""
    got = prefill_plan(steps, heads, kv, dim, q_f32, room=0)
    assert got["pair"] == pair and got["chunks"] == 1 and got["parts"] == 0


@pytest.mark.parametrize("steps,heads,kv,dim,q_f32,pair", [
    (8192, 8, 2, 256, False, True),    # 254 / 277
    (6000, 8, 2, 256, True, False),    # 260 / 235
    (8192, 16, 2, 128, False, True),   # 312 / 314
    (16384, 16, 2, 128, True, True),   # 1397 / 1443
    (7000, 32, 8, 128, True, True),    # 547 / 565
    (768, 32, 8, 128, False, False),   # 33.4 / 31.0
    (4500, 16, 2, 256, True, False),   # 306 / 242
])
def test_calls_with_partials_take_the_faster_kernel(steps, heads, kv, dim, q_f32, pair):
    assert prefill_plan(steps, heads, kv, dim, q_f32)["pair"] == pair


# us, query blocks by subset (0) against longest first over all subsets (2)
@pytest.mark.parametrize("steps,heads,kv,dim,q_f32,order", [
    (3001, 16, 2, 256, True, 0),   # 126.7 / 128.1
    (2600, 16, 2, 256, True, 0),   # 111.1 / 111.9
    (6000, 8, 2, 256, True, 0),    # 235.3 / 239.2
    (3504, 16, 2, 256, True, 0),   # the last with 219 query blocks
    (3505, 16, 2, 256, True, 2),
    (3584, 16, 2, 256, True, 2),   # 161.5 / 155.0
    (1500, 32, 8, 128, False, 2),  # 56.6 / 39.3, eight subsets
    (12000, 4, 4, 256, True, 2),   # 555 / 461, four
])
def test_order_of_whole_query_blocks(steps, heads, kv, dim, q_f32, order):
    got = prefill_plan(steps, heads, kv, dim, q_f32, room=0)
    assert (got["pair"], got["chunks"], got["order"]) == (0, 1, order)


@pytest.mark.parametrize("steps,heads,kv,dim,q_offset", [(4500, 8, 2, 256, 0), (3001, 32, 8, 128, 0), (4200, 8, 2, 256, 300)])
def test_cut_plan_has_room_for_the_cut_blocks_only(steps, heads, kv, dim, q_offset):
    """A longest-first grid that cuts query blocks in two keeps partials of those past the cut."""
    plan = prefill_plan(steps, heads, kv, dim, False, q_offset=q_offset)
    group = heads // kv
    pos = 16 * (8 // (group & -group))
    nqb, subsets = -(-steps // pos), kv * (group // (group & -group))
    blocks = [-(-(q_offset + min(steps, (b + 1) * pos)) // 64) for b in range(nqb)]
    if plan["order"] == 2 and plan["chunks"] == 2:
        cut = sum(n > plan["chunk"] for n in blocks)
        assert 0 < cut < nqb
        rows = subsets * cut * 2 * 128
    else:
        assert plan["chunks"] == 1
        rows = 0
    room = _lib.lib().bt_prefill_partials_bytes(steps, q_offset, heads, kv, dim)
    assert room == rows * (dim * 4 + 4)
    if rows:  # one byte less, and the plan is one without partials
        assert prefill_plan(steps, heads, kv, dim, False, room=room - 1, q_offset=q_offset)["chunks"] == 1


def test_plan_refuses_what_the_call_refuses():
    lib, out = _lib.lib(), (ctypes.c_int32 * 5)()
    assert lib.bt_prefill_plan(8, 0, 8, 2, 64, _lib.BT_DTYPE_F32, 0, ctypes.addressof(out)) == _lib.BT_ENOTSUP
    assert lib.bt_prefill_plan(0, 0, 8, 2, 256, _lib.BT_DTYPE_F32, 0, ctypes.addressof(out)) == _lib.BT_EINVAL
    assert lib.bt_prefill_plan(8, 0, 9, 2, 256, _lib.BT_DTYPE_F32, 0, ctypes.addressof(out)) == _lib.BT_EINVAL
    assert lib.bt_prefill_plan(8, 0, 8, 2, 256, 7, 0, ctypes.addressof(out)) == _lib.BT_EINVAL
    assert lib.bt_prefill_plan(8, 0, 8, 2, 256, _lib.BT_DTYPE_F32, 0, None) == _lib.BT_EINVAL
