"""The order of the squeeze-excite gate's f32 sums: the row chunks' sums added in chunk order from
the first, a squeeze output's terms c = lane, lane + 64, ... of a wave lane in order, an excite
output's terms in order of the squeeze outputs starting from the bias. A calibrated forward
quantizes what the gate scales, so a gate that differs in its last bit moves values across
rounding boundaries: the order is part of the result. Each case holds a large value, values that
are absorbed by it (40 against half an ulp of 64 at 2^30), and its negative, so that every other
order leaves the absorbed ones."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402

BIG = 2.0 ** 30


@pytest.mark.parametrize("C,S", [(32, 18), (96, 33), (480, 20), (1152, 48)])
def test_excite_terms_in_order_from_the_bias(C, S):
    x = torch.ones(2, C, 7, 7, device="cuda").contiguous(memory_format=torch.channels_last)
    w1, b1 = torch.zeros(S, C, device="cuda"), torch.full((S,), 40.0, device="cuda")  # z = silu(40) = 40
    w2, b2 = torch.ones(C, S, device="cuda"), torch.full((C,), BIG, device="cuda")
    w2[:, S - 1] = -BIG / 40
    gate = I.se_gate_nhwc(x, w1, b1, w2, b2)  # 2^30 + 40 + ... + 40 - 2^30 (the last product rounded, below 64) -> 0
    last = torch.tensor(-BIG / 40, dtype=torch.float32).double() * 40 + BIG
    want = torch.sigmoid(last)
    assert abs(float(last)) < 64
    assert torch.allclose(gate.double().cpu(), want.expand(2, C), atol=1e-6)


@pytest.mark.parametrize("C,HW", [(32, 12544), (96, 3136), (144, 784), (240, 784)])
def test_chunks_in_order(C, HW):
    """One pixel of each chunk holds a value: 2^30, 40, ..., 40, -2^30."""
    chunks = max(1, min(HW * C // 16384, HW, 64))
    rows = (HW + chunks - 1) // chunks
    used = (HW + rows - 1) // rows
    assert used > 4
    x = torch.zeros(1, HW, C, device="cuda")
    x[0, ::rows] = 40.0
    x[0, 0], x[0, (used - 1) * rows] = BIG, -BIG
    x = x.reshape(1, HW, 1, C).permute(0, 3, 1, 2)
    w1 = torch.zeros(4, C, device="cuda")
    w1[0, C // 2] = float(HW) / 40
    w2 = torch.zeros(C, 4, device="cuda")
    w2[:, 0] = 1.0
    gate = I.se_gate_nhwc(x, w1, None, w2, None)
    assert torch.equal(gate, torch.full_like(gate, 0.5))  # a pooled value of 0: z = 0


@pytest.mark.parametrize("C", [192, 480, 1152])
def test_squeeze_lanes_in_order(C):
    """Channels 0, 64 and 128 are one lane's terms: 2^30, 40, -2^30 in that order."""
    x = torch.ones(1, C, 1, 1, device="cuda").contiguous(memory_format=torch.channels_last)
    w1 = torch.zeros(8, C, device="cuda")
    w1[:, 0], w1[:, 64], w1[:, 128] = BIG, 40.0, -BIG
    w1[:, 4] = 1.0  # a lane of its own
    gate = I.se_gate_nhwc(x, w1, None, torch.ones(C, 8, device="cuda"), None)
    want = torch.sigmoid(8 * torch.nn.functional.silu(torch.ones((), dtype=torch.float64)))
    assert torch.allclose(gate.double().cpu(), want.expand(1, C), atol=1e-6)
