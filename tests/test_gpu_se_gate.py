"""The squeeze-excite gates at the edges of their kernel's loops: few and many channels and squeeze
outputs, more than one pass over channels, outputs and terms."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402


# one group of channels; fewer chunks, channels and outputs than a batch of loads, and more (256
# channels and four outputs a wave, eight chunks and terms); one pass of 1024 threads' channels, two
# and the second nearly empty (1152, 1280, 2052), past four (4100); 64 outputs of the waves' first pass
# and more (300, 9000)
@pytest.mark.parametrize("N,C,S,HW", [(1, 4, 1, 1), (3, 12, 3, 50), (2, 32, 8, 12544), (3, 96, 4, 3136), (2, 240, 10, 784),
                                      (2, 672, 28, 196), (5, 1152, 48, 49), (2, 1280, 49, 49), (2, 1284, 48, 7),
                                      (1, 2048, 60, 49), (1, 2052, 20, 9), (1, 4100, 17, 4), (1, 64, 300, 100),
                                      (1, 400, 9000, 5)])
@pytest.mark.parametrize("bias", [True, False])
def test_gate_of_float64(N, C, S, HW, bias):
    """Within the f32 sums' bound of the float64 gate; the product's maxima exactly."""
    print(f"se gate N={N} C={C} S={S} HW={HW} bias={bias}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(N + C + S + HW)
    rn = lambda *s: torch.randn(*s, generator=g, device="cuda")  # noqa: E731
    x = (rn(N, C, HW, 1) + 0.3).contiguous(memory_format=torch.channels_last)
    w1, w2 = rn(S, C) * C ** -0.5, rn(C, S) * S ** -0.5
    b1, b2 = (rn(S), rn(C)) if bias else (None, None)
    gate = I.se_gate_nhwc(x, w1, b1, w2, b2)
    xd, a1, a2 = x.double().flatten(2), w1.double().abs(), w2.double().abs()
    o1, o2 = (b.double() if bias else 0.0 for b in (b1 if bias else 0, b2 if bias else 0))
    z0 = xd.mean(2) @ w1.double().t() + o1
    z = z0 * torch.sigmoid(z0)
    want = torch.sigmoid(z @ w2.double().t() + o2)
    u = 2.0 ** -24
    # each sum's error by its length and the sum of magnitudes; SiLU's slope is below 1.1, sigmoid's
    # 0.25; the hardware exp2 and reciprocal within 8 u of a value (their argument's rounding included)
    dz = 1.1 * (C + HW + 2) * u * (xd.abs().mean(2) @ a1.t() + abs(o1)) + 8 * u * (z.abs() + z0.abs() * z.abs())
    dp = dz @ a2.t() + (S + 2) * u * (z.abs() @ a2.t() + abs(o2))
    pre = (z @ w2.double().t() + o2).abs()
    bound = 0.25 * dp + 8 * u * (1 + pre) * want
    assert ((gate.double() - want).abs() <= bound).all()
    parts, n = gate._bq_product_absmax[:2]
    assert parts[:n].max() == (x.flatten(2) * gate[:, :, None]).abs().max()
