"""Ragged decode with the default number of work-groups (``ragged_target``): a
batch on either side of the line between one round of work-groups and several,
and past one round, planned on the host and on the device."""

from __future__ import annotations

import pytest
import torch

from breezetoken_amd import workloads as wl
from oracle import attention as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,rounds", [(48, 1), (49, 2), (128, 2), (129, 3)])
def test_default_rounds_match_the_oracle(hip_backend, batch, rounds):
    one = hip_backend.num_cus // 2
    if one == 128:
        assert hip_backend.ragged_target(batch, 2) == rounds * one
    # One long sequence among short ones: its splits take the room left.
    lens = [1 + (i * 37) % 90 for i in range(batch)]
    lens[batch // 3] = 6001
    case = wl.c5_inputs(lens=lens)
    off = torch.tensor(case.offsets, dtype=torch.int64, device="cuda")
    n = torch.tensor(case.lens, dtype=torch.int32, device="cuda")
    args = (case.q.float().cuda(), case.k.cuda(), case.v.cuda(), off, n)
    host = hip_backend.attention_ragged(*args, case.lens, case.scale)
    device = hip_backend.attention_ragged(*args, None, case.scale)
    assert torch.equal(host, device)
    out = host.cpu()
    for b, (m, o) in enumerate(zip(case.lens, case.offsets)):
        ref = orc.torch_attention(case.q[b].float(), case.k[o : o + m].float(), case.v[o : o + m].float(), case.scale)
        err, cos = orc.compare(out[b].numpy(), ref.numpy())
        # both sides sum exp-weighted bf16 values in f32; q and P carry 16 bits
        assert err <= 2e-4 and cos >= 0.99999, (b, m, err, cos)
