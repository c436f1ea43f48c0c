"""attention_batched takes whole numbers for max_len only, of any size."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


def _args():
    g = torch.Generator(device="cuda").manual_seed(3)
    q = torch.randn(2, 8, 128, device="cuda", generator=g)
    k, v = (torch.randn(128, 2, 128, device="cuda", generator=g).to(torch.bfloat16) for _ in range(2))
    pos = torch.tensor([50, 63], dtype=torch.int32, device="cuda")
    return q, k, v, pos, torch.tensor([0, 64], dtype=torch.int64, device="cuda"), 128**-0.5


@pytest.mark.parametrize("max_len", [64.0, "64", None])
def test_other_types_are_refused(hip_backend, max_len):
    with pytest.raises(TypeError):
        hip_backend.attention_batched(*_args(), max_len)


def test_a_bound_past_32_bits_is_a_bound(hip_backend):
    few, many = (hip_backend.attention_batched(*_args(), n) for n in (64, 2**40))
    # the same sums in other groups; q and P carry 16 bits
    assert (few - many).abs().max().item() <= 2e-5
