"""The longest-first grid of the two-waves-per-SIMD prefill kernel: a grid with a
work-group per CU or more runs the query blocks of all head subsets longest
first, the longest ones cut in two where that evens the end.

bt_prefill_longest_first turns a work-group index into (subset, query block, chunk)
by the function that the kernel calls; its items must cover every chunk once, in
their order.  The GPU tests run the shapes that take the grid, whole and cut, and the
pair kernel for f32 q, and ask the library which of these each one takes."""

from __future__ import annotations

import ctypes

import pytest
import torch

from breezetoken_amd import _lib
from test_prefill_choice import ALL, prefill_plan

KB = 64


def _items(S, P0, heads, kv, kb):
    lib, out = _lib.lib(), (ctypes.c_int32 * 3)()
    total = lib.bt_prefill_longest_first(S, P0, heads, kv, kb, -1, ctypes.addressof(out))
    assert total > 0
    for item in range(total):
        assert lib.bt_prefill_longest_first(S, P0, heads, kv, kb, item, ctypes.addressof(out)) == total
        yield tuple(out)


@pytest.mark.parametrize("S,P0,heads,kv", [(4500, 0, 8, 2), (3001, 0, 16, 2), (3001, 0, 32, 8), (700, 3000, 24, 4),
                                           (1, 0, 40, 5), (2049, 63, 1, 1), (1500, 0, 6, 2), (130, 8000, 3, 1)])
def test_items_cover_every_chunk_once(S, P0, heads, kv):
    group = heads // kv
    sub = group & -group
    pos, ys = 16 * (8 // sub), kv * (group // sub)
    nqb, nkb = -(-S // pos), (P0 + S + KB - 1) // KB
    blocks = [(P0 + min(S, (qb + 1) * pos) + KB - 1) // KB for qb in range(nqb)]
    for kb in sorted({nkb, (nkb + 1) // 2, nkb * 3 // 4, max(1, nkb - 1)}):
        if kb < (nkb + 1) // 2 or kb < 1:
            continue
        got = [(qb, y, c) for y, qb, c in _items(S, P0, heads, kv, kb) if y >= 0]
        want = {(qb, y, c) for qb in range(nqb) for y in range(ys) for c in range(-(-blocks[qb] // kb))}
        assert len(got) == len(set(got)) and set(got) == want
        # Three runs, each from its longest item: first chunks longer than any second
        # one, second chunks, the other first chunks.
        length = {i: min(kb, blocks[i[0]] - i[2] * kb) for i in got}
        second = [i for i in got if i[2] == 1]
        at = got.index(second[0]) if second else len(got)
        runs = [got[:at], second, got[at + len(second):]]
        assert runs[0] + runs[1] + runs[2] == got
        for run in runs:
            assert all(length[a] >= length[b] for a, b in zip(run, run[1:]))
        if second:
            top = length[second[0]]
            assert all(length[i] >= min(top + 1, kb) for i in runs[0]) and all(length[i] <= top for i in runs[2])


def test_grid_query_refuses_bad_chunks():
    lib, out = _lib.lib(), (ctypes.c_int32 * 3)()
    for kb, item in ((31, -1), (65, -1), (64, 10**6)):  # 64 key blocks in all
        assert lib.bt_prefill_longest_first(4096, 0, 8, 2, kb, item, ctypes.addressof(out)) == _lib.BT_EINVAL
    assert lib.bt_prefill_longest_first(4096, 0, 9, 2, 64, -1, ctypes.addressof(out)) == _lib.BT_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim,steps,q_f32,path,unsplit", [
    (8, 2, 256, 4500, False, "cut", "subset"),    # 282 work-groups, the longest of 71 blocks
    (8, 2, 256, 4500, True, "cut", "subset"),
    (16, 2, 256, 3700, True, "longest", "longest"),  # 232 query blocks a subset: the order over both
    (32, 8, 128, 1500, False, "longest", "longest"),  # eight subsets
    (24, 4, 128, 1400, True, "longest", "longest"),   # three subsets of two heads a kv head
    (16, 2, 256, 1500, True, "pair", "pair"),
    (32, 8, 128, 700, True, "pair", "pair"),
])
def test_rows_match_the_oracle(hip_backend, heads, kv, dim, steps, q_f32, path, unsplit):
    if hip_backend.num_cus == 256:
        for room, want in ((ALL, path), (0, unsplit)):
            plan = prefill_plan(steps, heads, kv, dim, q_f32, room)
            kind = ("pair" if plan["pair"] else "cut" if plan["chunks"] == 2 and plan["order"] == 2 else
                    "longest" if plan["chunks"] == 1 and plan["order"] == 2 else
                    "subset" if plan["chunks"] == 1 and not plan["parts"] else "other")
            assert kind == want
    from oracle import attention as orc

    print(f"[prefill] H={heads} Hkv={kv} D={dim} S={steps} f32={q_f32}", flush=True)
    g = torch.Generator().manual_seed(steps + heads)
    q = torch.randn(steps, heads, dim, generator=g)
    q = q if q_f32 else q.to(torch.bfloat16)
    k = torch.randn(steps, kv, dim, generator=g).to(torch.bfloat16)
    v = torch.randn(steps, kv, dim, generator=g).to(torch.bfloat16)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out = hip_backend.attention_prefill(qd, kd, vd, dim**-0.5)
    whole = hip_backend.attention_prefill(qd, kd, vd, dim**-0.5, split_keys=False)
    ref = orc.torch_prefill_attention(q.float(), k.float(), v.float(), dim**-0.5)
    for got in (out, whole):
        err, cos = orc.compare(got.cpu().numpy(), ref.numpy())
        # P and V are rounded to fp16: 2^-12 of sums of |v| below 4, either sign
        assert err <= 2e-3 and cos >= 0.99999, (err, cos)


@pytest.mark.gpu
def test_cut_rows_behind_a_cached_prefix(hip_backend):
    """Query rows at positions 300.. of a longer cache, on the longest-first grid."""
    from oracle import attention as orc

    g = torch.Generator().manual_seed(5)
    steps, off = 4200, 300
    q = torch.randn(steps, 8, 256, generator=g).to(torch.bfloat16)
    k = torch.randn(off + steps, 2, 256, generator=g).to(torch.bfloat16)
    v = torch.randn(off + steps, 2, 256, generator=g).to(torch.bfloat16)
    out = hip_backend.attention_prefill(q.cuda(), k.cuda(), v.cuda(), 1 / 16, q_offset=off)
    ref = orc.torch_prefill_banded(q.float(), k.float(), v.float(), off, 1 / 16)
    err, cos = orc.compare(out.cpu().numpy(), ref.numpy())
    assert err <= 2e-3 and cos >= 0.99999, (err, cos)
