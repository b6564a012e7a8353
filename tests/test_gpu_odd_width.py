"""Linears of widths that no vector divides: the padded quantizer and copy against rows padded by torch."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402
from borch_amd._lib import check, lib  # noqa: E402


# each kernel's width range and its edge, rows whose start is not 16-byte aligned, one value,
# the two-read kernel past 8192
@pytest.mark.parametrize("M,K", [(1, 1), (3, 13), (70, 255), (5, 257), (33, 511), (9, 513), (130, 1023), (7, 1025),
                                 (1000, 1555), (4, 2049), (6, 4097), (2, 8191), (3, 8193), (2, 20001)])
def test_padded_rows(M, K):
    """The bytes and scales of quantizing the rows padded by torch, and the padded f32 copy."""
    print(f"padded rows M={M} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M * 31 + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    x[0, K - 1] = 0.5 * 127  # a row of half-integer quotients at its end
    if M > 2:
        x[2] = 0.0
    kp = I.round_up(max(K, 16), 16)
    want = torch.nn.functional.pad(x, (0, kp - K))
    q, s = I.quantize_rows_padded(x, kp)
    qw, sw = I.quantize_rows(want)
    assert torch.equal(s, sw) and torch.equal(q, qw)
    off = torch.empty(M * K + 1, device="cuda")[1:].view(M, K).copy_(x)  # 4-byte aligned only
    q2, s2 = I.quantize_rows_padded(off, kp)
    assert torch.equal(s2, sw) and torch.equal(q2, qw)
    y = torch.full((M, kp), 7.0, device="cuda")
    check(lib().bq_pad_rows_f32(off.data_ptr(), M, K, kp, y.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(y, want)


@pytest.mark.parametrize("M,K,N", [(1, 30, 17), (4, 1555, 64), (7, 100, 33), (64, 1001, 300), (200, 77, 50)])
@pytest.mark.parametrize("mode", ["w8a8", "w8a32"])
def test_linear_of_odd_width(M, K, N, mode):
    """An odd-width Linear equals the same Linear on rows padded by torch to the packed width."""
    print(f"odd width {mode} M={M} K={K} N={N}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(K + N)
    x, w, b = (torch.randn(*s, generator=g, device="cuda") for s in ((M, K), (N, K), (N,)))
    kp = I.round_up(K, 16)
    w8 = I.pack_linear_weight(w, weight_only=mode == "w8a32")
    wide = I.Int8Weight(w8.q, w8.s, kp, N, w8.weight_only)
    xp = torch.nn.functional.pad(x, (0, kp - K))
    r = torch.randn(M, N, generator=g, device="cuda")
    assert torch.equal(I.linear(x, w8, b, I.ACT_RELU, r), I.linear(xp, wide, b, I.ACT_RELU, r))
    assert torch.equal(I.linear(x.expand(2, M, K), w8, b), I.linear(xp.expand(2, M, kp), wide, b))
