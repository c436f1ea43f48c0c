"""bt_ragged_plan_rounds on the host: one round of work-groups where it is even,
more where it is not, and otherwise exactly bt_ragged_plan."""

from __future__ import annotations

import ctypes

import pytest

from breezetoken_amd import _lib


def plan_rounds(lens, one, target):
    """(entries, work, base, count, total) of bt_ragged_plan_rounds."""
    b = len(lens)
    cap = max(b, one, target)
    arr = (ctypes.c_int32 * b)(*lens)
    work, base, cnt = (ctypes.c_int32 * (4 * cap))(), (ctypes.c_int32 * b)(), (ctypes.c_int32 * b)()
    tot = ctypes.c_int32()
    n = _lib.lib().bt_ragged_plan_rounds(ctypes.addressof(arr), b, one, target, ctypes.addressof(work), cap,
                                         ctypes.addressof(base), ctypes.addressof(cnt), ctypes.addressof(tot))
    return n, list(work)[: 4 * max(n, 0)], list(base), list(cnt), tot.value


@pytest.mark.parametrize("lens,one,target,many", [
    ([1000] * 96, 128, 256, False),           # 96 of 128: a third of a round idle at most
    ([1000] * 144, 128, 384, True),           # 144 take two rounds of 128
    ([1000] * 200, 128, 384, False),          # 200 nearly fill two
    ([20000] + [300] * 95, 128, 256, True),   # its 33 splits of 625 tokens against a mean of 380
    ([0] * 9, 4, 8, False),
])
def test_rounds_plan_is_one_of_two(lens, one, target, many):
    got = plan_rounds(lens, one, target)
    assert got == plan_rounds(lens, *([target] * 2 if many else [one] * 2))


def test_rounds_plan_refuses_bad_sizes():
    assert plan_rounds([5], 0, 4)[0] == _lib.BT_EINVAL
    assert plan_rounds([5], 4, 0)[0] == _lib.BT_EINVAL
