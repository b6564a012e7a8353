"""bq_attention_f32's bf16-piece products at the edges of its key blocks and query tiles, and on
non-finite inputs, against float64."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402


def _ref(x, H):
    B, T, D3 = x.shape
    q, k, v = x.double().reshape(B, T, 3, H, 64).permute(2, 0, 3, 1, 4).contiguous()
    p = torch.softmax(q @ k.transpose(-1, -2).contiguous() / 8, -1)
    s = (q.abs() @ k.abs().transpose(-1, -2).contiguous() / 8).amax(-1)  # scale of a score's rounding
    y = p @ v
    err = p @ v.abs()
    flat = [t.transpose(1, 2).reshape(B, T, D3 // 3) for t in (y, err, s[..., None].expand_as(y))]
    return flat


# one and 16 keys, each kernel's last full block and the next key, an odd block count's
# 16-key remainder (193..208), query tiles that end a wave early
@pytest.mark.parametrize("B,T,H", [(1, 1, 2), (3, 16, 1), (2, 33, 3), (1, 64, 5), (2, 65, 2), (1, 128, 3), (2, 129, 1),
                                   (1, 176, 2), (1, 193, 3), (2, 208, 2), (1, 209, 2), (1, 255, 3), (2, 256, 2)])
@pytest.mark.parametrize("scale", [0.1, 1.0, 8.0])
def test_pieces(B, T, H, scale):
    """Within the f32 bound of the two products and the softmax: a score is off by at most
    (64 + 2) 2^-24 of its sum of absolute products (and the pieces left out, 2^-26 more), which
    moves its exponential by that much relative, as does the maximum it is taken from; the
    exponential, the sums over T keys and the division add (T + 8) 2^-24 of sum p |v|."""
    print(f"attention pieces B={B} T={T} H={H} scale={scale}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(T + H)
    x = torch.randn(B, T, 3 * 64 * H, generator=g, device="cuda") * scale
    y, mag, s = _ref(x, H)
    bound = (2 * (64 + 3) * 2.0 ** -24 * s * 2 + (T + 8) * 2.0 ** -24) * mag + 1e-30
    err = (I.attention_f32(x, H).double() - y).abs()
    assert bool((err <= bound).all()), f"max err / bound {float((err / bound).max())}"


def test_non_finite():
    """An infinite or NaN value reaches the outputs that f32 arithmetic gives it, and no others:
    v's infinity its head dim, k's -inf score a zero weight, q's NaN its own row."""
    g = torch.Generator(device="cuda").manual_seed(3)
    B, T, H = 2, 197, 2
    x = torch.randn(B, T, 3, H, 64, generator=g, device="cuda")
    x[0, :, 0, 0, 5] = x[0, :, 0, 0, 5].abs() + 0.1  # q's dim 5 positive, so k's -inf there scores -inf
    x[0, 7, 1, 0, 5] = -float("inf")
    x[0, 3, 2, 1, 9] = float("inf")
    x[1, 4, 0, 0, 0] = float("nan")
    x[1, 9, 2, 1, 1] = 3.4e38
    clean = x.clone()
    clean[0, 3, 2, 1, 9] = 0.0
    y = I.attention_f32(x.reshape(B, T, -1).contiguous(), H).reshape(B, T, H, 64)
    want = _ref(x.reshape(B, T, -1), H)[0].reshape(B, T, H, 64)
    assert torch.equal(torch.isnan(y), torch.isnan(want))
    assert torch.equal(torch.isinf(y), torch.isinf(want)) and bool((y[0, :, 1, 9] == float("inf")).all())
    ok = torch.isfinite(want)
    assert int((~ok).sum()) == T + 64
    assert torch.allclose(y[ok].double(), want[ok], rtol=1e-4, atol=1e-5)
    rest = I.attention_f32(clean.reshape(B, T, -1).contiguous(), H).reshape(B, T, H, 64)
    assert torch.equal(torch.isfinite(rest[0]), torch.ones_like(rest[0], dtype=torch.bool))
