"""The decode matvec at the edges of its two kernels' shapes, against float64."""

from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize(
    "K,N",
    [(255, 3072), (256, 3072), (257, 3080), (512, 8192), (512, 8200), (513, 6144), (1000, 6152), (1024, 8200),
     (1025, 8200), (1025, 12288), (1024, 12280), (1536, 24576), (1535, 24584), (300, 65536), (300, 65544),
     (1025, 4096), (1031, 4088), (2048, 4104), (2049, 128), (2056, 1000), (2304, 7168), (2304, 32768), (2305, 32776),
     (4096, 8), (4099, 2056), (5119, 5128), (6143, 2048), (6144, 2048), (16384, 264)],
)
def test_matvec_at_shape_edges(hip_backend, K, N):
    gen = torch.Generator(device="cuda").manual_seed(K * 7 + N)
    # A wider matrix, whose other columns must not be read into the results.
    wide = torch.full((K, N + 8), float("nan"), device="cuda", dtype=torch.bfloat16)
    wide[:, :N] = torch.randn(K, N, device="cuda", generator=gen).to(torch.bfloat16)
    w = wide[:, :N]
    x = torch.randn(K, device="cuda", generator=gen)
    ref = x.double() @ w.double()
    # Rows of one lane, its passes, the lanes, the waves and at most 64 shares are
    # added in turn: under 192 roundings of 2^-24 on any term's way.
    bound = 192 * 2.0**-24 * (x.double().abs() @ w.double().abs())
    for m in (w, w.contiguous()):
        y = hip_backend.linear(x, m).double()
        assert ((y - ref).abs() <= bound).all()
