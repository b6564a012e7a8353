"""bq_attention_f32's error against float64 as a whole (2-norm), over score scales: no larger than f32
products and sums (f32 MFMAs) came out with at the same sizes."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402


# (tokens, scale of q and k): the error of f32 MFMAs on these inputs
F32 = {(64, 0.1): 1.15e-7, (64, 1.0): 2.60e-7, (64, 8.0): 1.85e-6, (130, 0.1): 1.55e-7, (130, 1.0): 2.97e-7,
       (130, 8.0): 2.17e-6, (197, 0.1): 1.92e-7, (197, 1.0): 3.26e-7, (197, 8.0): 2.23e-6, (256, 0.1): 2.17e-7,
       (256, 1.0): 3.48e-7, (256, 8.0): 2.48e-6}


@pytest.mark.parametrize("T,scale", sorted(F32))
def test_no_further_from_float64_than_f32(T, scale):
    err = ref = 0.0
    for seed in range(4):
        g = torch.Generator(device="cuda").manual_seed(seed)
        x = torch.randn(4, T, 3, 3, 64, generator=g, device="cuda")
        x[:, :, :2] *= scale
        q, k, v = (t.transpose(1, 2).contiguous() for t in x.double().unbind(2))
        want = (torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) / 8, -1) @ v).transpose(1, 2)
        y = I.attention_f32(x.reshape(4, T, -1).contiguous(), 3).reshape(4, T, 3, 64)
        err += float((y.double() - want).norm()) ** 2
        ref += float(want.norm()) ** 2
    assert (err / ref) ** 0.5 < F32[T, scale]
