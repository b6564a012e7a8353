"""bq_attention_f32 where the scores are so large that a softmax has one key left, or few: the
exponential of the largest score is 1 whatever its size."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402


@pytest.mark.parametrize("T", [17, 64, 197, 256])
@pytest.mark.parametrize("lo,hi", [(3e2, 5e2), (1.2e4, 2.1e4), (2e5, 9e5), (1e9, 4e9)])
def test_one_key_left(T, lo, hi):
    """Rows of sign patterns with magnitudes in lo .. hi: raw scores up to 64 hi^2, the best key's
    far above the next. Its weight is 1 and the others' 0, so the output is its v, bit for bit (a
    value is the sum of its pieces in any order that adds the small ones first)."""
    print(f"attention large scores T={T} {lo}..{hi}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T)
    B, H = 4, 3
    sign = torch.where(torch.rand(B, T, H, 64, generator=g, device="cuda") < 0.5, -1.0, 1.0)
    mag = lambda: lo + (hi - lo) * torch.rand(B, T, H, 1, generator=g, device="cuda")  # noqa: E731
    q, k = sign * mag(), sign * mag()
    v = torch.randn(B, T, H, 64, generator=g, device="cuda")
    s = torch.matmul(q.double().transpose(1, 2).contiguous(), k.double().permute(0, 2, 3, 1).contiguous()) / 8
    top, at = s.topk(2, -1)
    assert float((top[..., 0] - top[..., 1]).min()) > 200  # exp(-200) is 0 in f32
    y = I.attention_f32(torch.stack([q, k, v], 2).reshape(B, T, 3 * 64 * H).contiguous(), H).reshape(B, T, H, 64)
    want = torch.gather(v.transpose(1, 2), 2, at[..., :1].expand(B, H, T, 64)).transpose(1, 2)
    assert torch.equal(y, want)


@pytest.mark.parametrize("scale", [1.0, 3.5e4, 4.5e4, 6e4, 3e8])
def test_equal_scores(scale):
    """Equal keys have equal weights: the outputs are v's mean within the f32 sum's bound."""
    g = torch.Generator(device="cuda").manual_seed(5)
    B, T, H = 2, 197, 2
    q = torch.randn(B, T, H, 64, generator=g, device="cuda") * scale
    k = (torch.randn(B, 1, H, 64, generator=g, device="cuda") * scale).expand(B, T, H, 64)
    v = torch.randn(B, T, H, 64, generator=g, device="cuda")
    y = I.attention_f32(torch.stack([q, k, v], 2).reshape(B, T, 3 * 64 * H).contiguous(), H).reshape(B, T, H, 64)
    want = v.double().mean(1, keepdim=True).expand(B, T, H, 64)
    bound = (T + 8) * 2.0 ** -24 * v.double().abs().mean(1, keepdim=True)
    assert bool(((y.double() - want).abs() <= bound).all())
