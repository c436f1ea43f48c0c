"""The longest-first grid of the two-waves-per-SIMD prefill kernel: a grid with a
work-group per CU or more runs the query blocks of all head subsets longest
first, the longest ones cut in two where that evens the end.

The device code (gqa_prefill8.hip: split_compact = 2) turns a work-group index
into (query block, subset, chunk); the arithmetic is restated here and must
cover every item once, longest first within each region.  The GPU tests run the
shapes that take the grid, whole and cut, and those whose kernel the estimate
of capi.hip now chooses (the pair kernel for f32 q from about 1,500 tokens)."""

from __future__ import annotations

import pytest
import torch

KB = 64


def _past(c, kb, S, P0, pos, nqb):
    R = c * kb * KB - P0
    if R < 0:
        return nqb
    return 0 if S <= R else nqb - R // pos


def _items(kb, S, P0, pos, ys):
    nqb = -(-S // pos)
    nkb = (P0 + S + KB - 1) // KB
    chunks = -(-nkb // kb)
    assert chunks <= 2
    ahead = _past(1, nkb - kb, S, P0, pos, nqb) if chunks > 1 and nkb > kb else nqb
    second = _past(1, kb, S, P0, pos, nqb) if chunks > 1 else 0
    pad = lambda n: (n + 7) // 8 * 8  # noqa: E731
    end0 = pad(ahead * ys)
    end1 = end0 + pad(second * ys)
    total = end1 + pad((nqb - ahead) * ys)
    for L in range(total):
        if L >= end1:
            at, items, rank, chunk = L - end1, (nqb - ahead) * ys, ahead, 0
        elif L >= end0:
            at, items, rank, chunk = L - end0, second * ys, 0, 1
        else:
            at, items, rank, chunk = L, ahead * ys, 0, 0
        if at < items:
            yield nqb - 1 - rank - at // ys, at % ys, chunk


@pytest.mark.parametrize("S,P0,pos,ys", [(4500, 0, 32, 2), (3001, 0, 16, 2), (3001, 0, 32, 8), (700, 3000, 16, 3),
                                         (1, 0, 16, 5), (2049, 63, 128, 1)])
def test_items_cover_every_chunk_once(S, P0, pos, ys):
    nqb, nkb = -(-S // pos), (P0 + S + KB - 1) // KB
    blocks = lambda qb: (P0 + min(S, (qb + 1) * pos) + KB - 1) // KB  # noqa: E731
    for kb in sorted({nkb, (nkb + 1) // 2, nkb * 3 // 4, max(1, nkb - 1)}):
        if kb < (nkb + 1) // 2 or kb < 1:
            continue
        got = list(_items(kb, S, P0, pos, ys))
        want = {(qb, y, c) for qb in range(nqb) for y in range(ys) for c in range(-(-blocks(qb) // kb))}
        assert len(got) == len(set(got)) and set(got) == want
        # no item starts behind one shorter than half of it (the regions' order)
        length = [min(kb, blocks(qb) - c * kb) for qb, _, c in got]
        assert all(a >= b for a, b in zip(length, length[1:]) if a >= nkb - kb > b or a >= kb)


@pytest.mark.gpu
@pytest.mark.parametrize("heads,kv,dim,steps,q_f32", [
    (8, 2, 256, 4500, False),    # cut: 282 work-groups, the longest of 71 blocks
    (8, 2, 256, 4500, True),
    (32, 8, 128, 1500, False),   # whole, eight subsets
    (24, 4, 128, 1400, True),    # three subsets of two heads a kv head
    (16, 2, 256, 1500, True),    # pair kernel
    (32, 8, 128, 700, True),     # pair kernel, D = 128
])
def test_rows_match_the_oracle(hip_backend, heads, kv, dim, steps, q_f32):
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
