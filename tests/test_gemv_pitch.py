"""The matvec's choice of kernel by where W's rows lie (bt_gemv_plan), and its results on
both sides of each line, in room of exactly bt_gemv_workspace_bytes."""

from __future__ import annotations

import ctypes

import pytest
import torch

from breezetoken_amd import _lib


def plan(K, N, ldw, base=1 << 20):
    out = (ctypes.c_int32 * 3)()
    _lib.check("bt_gemv_plan", _lib.lib().bt_gemv_plan(base, ldw, K, N, ctypes.addressof(out)))
    return tuple(out)


# us, column kernel / strips
@pytest.mark.parametrize("K,N,ldw,base,strips", [
    (1536, 16392, 16392, 0, False),   # 13.1 / 16.1: rows not on a line
    (3072, 16392, 16392, 0, False),   # 21.7 / 25.8
    (2560, 1024, 1032, 0, False),     # 6.35 / 6.53
    (2560, 1024, 1088, 0, True),      # 6.22 / 5.84, on a line
    (2560, 1024, 1088, 64, False),    # its base is not
    (4096, 4104, 4104, 0, False),     # 12.1 / 12.6
    (16384, 2056, 2056, 0, False),    # 19.3 / 21.6
    (5120, 1032, 1032, 0, True),      # 9.2 / 7.2
    (5120, 3000, 3000, 0, True),      # 13.5 / 11.0
    (8192, 1672, 1672, 0, True),      # 15.1 / 10.5: seven tiles do not fill a round
    (8192, 2048, 2056, 0, False),     # eight do
    (2304, 4104, 4104, 0, True),      # 9.9 / 8.9
    (6144, 5128, 5128, 0, True),      # 22.5 / 19.3
    (5120, 2056, 2056, 0, True),      # 12.1 / 9.6
    (512, 16392, 16392, 0, True),     # 0.79 of the column kernel's time
    (512, 65528, 65528, 0, False),    # 1.08
    (768, 6152, 6152, 0, True),       # 0.91
    (1024, 8184, 8184, 0, False),     # 1.03
    (1024, 19432, 19432, 0, True),    # 14.4 / 12.3
    (1024, 6176, 6176, 0, True),      # 0.88: half a line, strips of 32 columns
    (1280, 16448, 16448, 0, True),    # 0.84: 128.5 lines
    (12288, 2040, 2048, 0, False),    # 13.1 / 13.9: rows of 4 KB
    (12288, 2048, 2048, 0, False),    # 12.5 / 13.8
    (8453, 1936, 2048, 0, False),     # 11.3 / 12.1
    (8453, 1600, 2048, 0, True),      # 13.4 / 9.4: not a full round of the column kernel
    (6144, 2048, 2048, 0, False),     # 8.73 / 8.95
    (6144, 2040, 2048, 0, True),      # 9.21 / 8.96
    (7000, 2048, 2048, 0, True),      # 10.7 / 9.3
    (8192, 2048, 2048, 0, True),      # 12.1 / 9.9
    (10240, 2048, 4096, 0, False),    # 11.9 / 14.5, 8 KB
    (16384, 2048, 4096, 0, True),     # 23.7 / 18.6
    (12288, 2048, 2112, 0, True),     # 12.1 / 12.0
    (8192, 4096, 4096, 0, True),      # 17.2 / 14.9
])
def test_kernel_by_rows_of_w(K, N, ldw, base, strips):
    assert plan(K, N, ldw, (1 << 20) + base)[0] == strips


@pytest.mark.parametrize("K", [1, 255, 256, 512, 513, 769, 1024, 1536, 2049, 4096, 6144, 8192, 16384])
@pytest.mark.parametrize("N", [8, 264, 1024, 2048, 3080, 6144, 8200, 16392, 20008, 65528, 131072])
def test_workspace_holds_either_plan(K, N):
    room = _lib.lib().bt_gemv_workspace_bytes(K, N)
    for ldw in (N, -(-N // 64) * 64, -(-N // 2048) * 2048, -(-N // 4096) * 4096 + 8):
        for base in (0, 16, 64):
            splits = plan(K, N, ldw, (1 << 20) + base)[2]
            assert (splits * N * 4 if splits > 1 else 0) <= room


def test_plan_refuses_what_the_call_refuses():
    out = (ctypes.c_int32 * 3)()
    call = lambda *a: _lib.lib().bt_gemv_plan(*a, ctypes.addressof(out))  # noqa: E731
    assert call(1 << 20, 1020, 1024, 1024) == _lib.BT_EINVAL
    assert call((1 << 20) + 8, 1024, 1024, 1024) == _lib.BT_EINVAL
    assert call(1 << 20, 1024, 1024, 1020) == _lib.BT_EINVAL


@pytest.mark.gpu
@pytest.mark.parametrize("K,N", [(512, 57344), (512, 57352), (1024, 32768), (1025, 18440), (768, 6152), (2056, 8184), (776, 6152), (4096, 3000), (8191, 2056), (8192, 2056),
                                 (4607, 1000), (4608, 1536), (4608, 1544), (6144, 1032), (6143, 2048), (6144, 2048), (8192, 1800),
                                 (8193, 2048), (10240, 2040)])
def test_results_at_each_pitch(hip_backend, K, N):
    gen = torch.Generator(device="cuda").manual_seed(K + N)
    x = torch.randn(K, device="cuda", generator=gen)
    w = torch.randn(K, N, device="cuda", generator=gen).to(torch.bfloat16)
    ref = x.double() @ w.double()
    # as in test_gemv_strips_gpu: under 192 roundings of 2^-24 on any term's way
    bound = 192 * 2.0**-24 * (x.double().abs() @ w.double().abs())
    for ldw in sorted({N, -(-N // 64) * 64, -(-N // 2048) * 2048}):
        for shift in (0, 8):  # of the base, in columns
            flat = torch.full((K * ldw + 8,), float("nan"), device="cuda", dtype=torch.bfloat16)
            view = flat[shift : shift + K * ldw].view(K, ldw)[:, :N]
            view.copy_(w)
            y = hip_backend.linear(x, view).double()
            assert ((y - ref).abs() <= bound).all(), (ldw, shift)
