"""bq_attention_f32 on values whose bf16 pieces fall below bf16's last bit."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402


@pytest.mark.parametrize("T", [5, 64, 197, 256])
@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -112, 2.0 ** -118, 2.0 ** -122])
def test_tiny_v(T, scale):
    """One head's v scaled down to the smallest normal numbers, another's zero: the first as close
    to float64 as ordinary values come (3e-7 as a whole, below 1e-6), the second zero, the third
    head's bits those of a call on ordinary values."""
    g = torch.Generator(device="cuda").manual_seed(T)
    B, H = 2, 3
    x = torch.randn(B, T, 3, H, 64, generator=g, device="cuda")
    plain = I.attention_f32(x.reshape(B, T, -1).contiguous(), H).reshape(B, T, H, 64)
    x[:, :, 2, 0] *= scale
    x[:, :, 2, 1] = 0
    y = I.attention_f32(x.reshape(B, T, -1).contiguous(), H).reshape(B, T, H, 64)
    q, k, v = x[:, :, :, 0].double().permute(2, 0, 1, 3).contiguous()
    want = torch.softmax(q @ k.transpose(-1, -2).contiguous() / 8, -1) @ v
    assert float((y[:, :, 0].double() - want).norm() / want.norm()) < 1e-6
    assert not bool(y[:, :, 1].any())
    assert torch.equal(y[:, :, 2], plain[:, :, 2])
