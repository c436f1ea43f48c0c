"""Decode by device position over caches on both sides of the slot count from which
K is read in whole rows (D = 256, more than 4 heads a kv head): there the two forms
give the same bits.  The other shapes read K one way at either size; they are checked
against the oracle, as these are, and that nothing past the position counts."""

from __future__ import annotations

import pytest
import torch

from oracle import attention as orc

pytestmark = pytest.mark.gpu

SLOTS = 16384


@pytest.mark.parametrize("heads,kv,dim", [(16, 2, 256), (10, 2, 256), (8, 2, 256), (16, 2, 128), (6, 3, 64)])
@pytest.mark.parametrize("valid", [1, 15, 16, 17, 2049, 16371, SLOTS - 1])
@pytest.mark.parametrize("q_dtype", [torch.float32, torch.bfloat16])
def test_rows_and_pieces_agree(hip_backend, heads, kv, dim, valid, q_dtype):
    gen = torch.Generator(device="cuda").manual_seed(valid + dim)
    q = torch.randn(heads, dim, device="cuda", generator=gen).to(q_dtype)
    k, v = (torch.full((SLOTS, kv, dim), float("nan"), device="cuda", dtype=torch.bfloat16) for _ in range(2))
    for c in (k, v):
        c[:valid] = torch.randn(valid, kv, dim, device="cuda", generator=gen).to(torch.bfloat16)
    pos = torch.tensor([valid - 1], dtype=torch.int32, device="cuda")
    scale = dim**-0.5
    least = hip_backend.attention_fixed(q, k, v, pos, scale)
    fewer = hip_backend.attention_fixed(q, k[: SLOTS - 1], v[: SLOTS - 1], pos, scale)
    ref = orc.torch_attention(q.float().cpu(), k[:valid].float().cpu(), v[:valid].float().cpu(), scale)
    for out in (least, fewer):
        err, cos = orc.compare(out.float().cpu().numpy(), ref.numpy())
        # q and P carry 16 bits, sums are f32: 2^-16 of |v| sums to about 1e-4 at most
        assert err <= 2e-4 and cos >= 0.999999, (err, cos)
    if dim == 256 and heads // kv > 4:
        assert torch.equal(least, fewer)  # whole rows and pieces: the same products in the same order
    else:
        # one form for both, in splits of the same tiles; 2^-16 relative in q and P
        assert (least - fewer).abs().max().item() <= 2e-5
