"""bt_ragged_plan_cost: short sequences keep one round of work-groups where further splits
cost more than they shorten, on the host and on the device."""

from __future__ import annotations

import ctypes

import pytest
import torch

from breezetoken_amd import _lib
from test_ragged_rounds import plan_rounds


def plan_cost(lens, one, target, tokens):
    """(entries, work, base, count, total) of bt_ragged_plan_cost."""
    b, cap = len(lens), max(len(lens), one, target)
    arr = (ctypes.c_int32 * b)(*lens)
    work, base, cnt = (ctypes.c_int32 * (4 * cap))(), (ctypes.c_int32 * b)(), (ctypes.c_int32 * b)()
    tot = ctypes.c_int32()
    n = _lib.lib().bt_ragged_plan_cost(ctypes.addressof(arr), b, one, target, tokens, ctypes.addressof(work), cap,
                                       ctypes.addressof(base), ctypes.addressof(cnt), ctypes.addressof(tot))
    return n, list(work)[: 4 * max(n, 0)], list(base), list(cnt), tot.value


def _lens(batch, lo, hi, seed=0):
    u = torch.rand(batch, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    return [int(lo * (hi / lo) ** float(x)) for x in u]


CASES = {
    "short_d256": (_lens(144, 32, 300), 128, 384, 300, False),
    "short_d128": (_lens(24, 32, 300), 32, 96, 150, False),
    "long_d256": (_lens(144, 256, 32768), 128, 384, 300, True),
    "long_d64": (_lens(200, 256, 4000), 128, 384, 120, True),
    "one_long": ([20000] + [300] * 95, 128, 256, 150, True),
    "even": ([1000] * 96, 128, 256, 1, False),
    "just_pays": ([64] * 5, 4, 10, 25, True),  # 5 x 64 -> 10 x 32: 25 * 5 <= 32 * 4
    "just_not": ([64] * 5, 4, 10, 26, False),
    "sorted_600": (_lens(600, 1, 900), 128, 1024, 300, False),
    "narrow_900": (_lens(900, 1, 9000), 128, 1408, 100, True),
}


@pytest.mark.parametrize("name", list(CASES))
def test_cost_plan_is_one_of_two(name):
    lens, one, target, tokens, many = CASES[name]
    assert plan_cost(lens, one, target, tokens) == plan_rounds(lens, *([target] * 2 if many else [one] * 2))
    assert plan_cost(lens, one, target, 0) == plan_rounds(lens, one, target)


def test_cost_plan_refuses_a_negative_cost():
    assert plan_cost([5], 4, 8, -1)[0] == _lib.BT_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("name", list(CASES))
def test_device_cost_plan_equals_host_plan(hip_backend, name):
    lens, one, target, tokens, _ = CASES[name]
    print(f"[plan] {name}: batch {len(lens)}", flush=True)
    n, work_h, base_h, cnt_h, tot = plan_cost(lens, one, target, tokens)
    seq_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
    work, cap, base, cnt, _ = hip_backend.ragged_plan_device(seq_len, target, one, tokens)
    assert base.cpu().tolist() == base_h and cnt.cpu().tolist() == cnt_h
    w = work.cpu().reshape(-1).tolist()
    assert w[: 4 * tot] == work_h and w[4 * tot :] == [-1, 0, 0, 0] * (cap - tot)
