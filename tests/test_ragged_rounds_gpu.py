"""Ragged decode with the default number of work-groups (``ragged_groups``): a
batch on either side of the line between one round of work-groups and several,
and past one round, planned on the host and on the device."""

from __future__ import annotations

import pytest
import torch

from breezetoken_amd import workloads as wl
from oracle import attention as orc
from test_ragged_rounds import plan_rounds

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,rounds", [(48, 1), (49, 2), (128, 2), (129, 3)])
def test_default_rounds_match_the_oracle(hip_backend, batch, rounds):
    one = hip_backend.num_cus // 2
    if one == 128:
        assert hip_backend.ragged_groups(batch, 2) == (one, rounds * one)
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


def _lens(batch, lo, hi, seed=0):
    u = torch.rand(batch, generator=torch.Generator().manual_seed(seed), dtype=torch.float64)
    return [int(lo * (hi / lo) ** float(x)) for x in u]


ROUND_CASES = {
    "even": ([1000] * 96, 128, 256),
    "uneven": (_lens(144, 256, 32768), 128, 384),
    "empty": ([0] * 70, 8, 64),
    "one": ([1], 1, 5),
    "counted_256": (_lens(256, 1, 20000), 128, 384),
    "sorted_257": (_lens(257, 1, 20000), 128, 384),
    "sorted_ties": ([64, 1000, 64, 33] * 100, 16, 64),
    "wide_candidates_512": (_lens(512, 1, 20000), 128, 1024),
    "narrow_candidates_513": (_lens(513, 1, 20000), 128, 1024),
    "scan_passes_1025": (_lens(1025, 1, 4000), 128, 1408),
    "largest_batch": (_lens(4096, 1, 300), 256, 4608),
    "longest_lengths": ([2**31 - 1, 2**31 - 2, 5, 2**30], 128, 256),
}


@pytest.mark.parametrize("name", list(ROUND_CASES))
def test_device_rounds_plan_equals_host_plan(hip_backend, name):
    """Both planners pick the same size and build the same tables, over the search's and the
    scan's steps; only the plan runs (no cache of these lengths exists)."""
    lens, one, target = ROUND_CASES[name]
    print(f"[plan] {name}: batch {len(lens)}", flush=True)
    n, work_h, base_h, cnt_h, tot = plan_rounds(lens, one, target)
    seq_len = torch.tensor(lens, dtype=torch.int32, device="cuda")
    work, cap, base, cnt, _ = hip_backend.ragged_plan_device(seq_len, target, one)
    torch.cuda.synchronize()
    assert base.cpu().tolist() == base_h and cnt.cpu().tolist() == cnt_h
    w = work.cpu().reshape(-1).tolist()
    assert w[: 4 * tot] == work_h
    assert w[4 * tot :] == [-1, 0, 0, 0] * (cap - tot)
