"""The weight-only Linear at the ends of its value and size ranges, in every kernel: empty products,
sums that overflow before their scale, infinite scales."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402
from borch_amd._lib import check, lib  # noqa: E402

INF = float("inf")


def _packed(q, s):
    return I.Int8Weight(q.to(torch.int8).contiguous(), s.contiguous(), q.shape[1], q.shape[0], True)


@pytest.mark.parametrize("M,N", [(3, 40), (8, 17), (40, 300), (600, 4099)])
def test_empty_product(M, N):
    """K = 0 through the C entries: act(bias + residual)."""
    print(f"w8a32 K=0 M={M} N={N}", flush=True)
    b, r = torch.randn(N, device="cuda"), torch.randn(M, N, device="cuda")
    pad = torch.empty(16, device="cuda")  # x and W are 16-byte aligned pointers that nothing is read from
    st = torch.cuda.current_stream().cuda_stream
    out = torch.full((M, N), 7.0, device="cuda")
    check(lib().bq_linear_w8a32(pad.data_ptr(), pad.data_ptr(), M, N, 0, b.data_ptr(), b.data_ptr(), r.data_ptr(),
                                I.ACT_RELU, out.data_ptr(), st))
    assert torch.equal(out, torch.relu(b + r))


# rows of the GEMV, the f32-MFMA kernel, the K-split one's forms (four waves at K = 272) and the
# tiled one's: 64 x 64, 64 x 128 and 128 x 128 workgroups, each with ragged columns and K
SHAPES = [(4, 64, 1024), (8, 64, 1024), (6, 300, 4096), (16, 4096, 4112), (16, 2048, 8208), (20, 768, 3072), (40, 2051, 2064), (100, 300, 272),
          (256, 3072, 1040), (700, 2051, 592), (600, 4099, 144), (1700, 2051, 144)]


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_sums_that_overflow_before_their_scale(M, N, K):
    """x * q sums past f32's range while x * (q * s) stays in it: finite, as the effective weights'
    products give it. Every third row is of ordinary size."""
    print(f"w8a32 large x M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda")
    q = torch.randint(-127, 128, (N, K), generator=g, device="cuda")
    s = (0.5 + torch.rand(N, generator=g, device="cuda")) / 127
    big = torch.arange(M, device="cuda") % 3 != 0
    x[big, 0] = 3.0e36
    q[:, 0] = 127 - torch.arange(N, device="cuda") % 40  # x * q is past 2.6e38, or near it, from the first value on
    x[big, 1:] *= 1e30
    w8 = _packed(q, s)
    y = I.linear_w8a32(x, w8)
    wd = q.double() * s.double()[:, None]
    want = x.double() @ wd.t()
    assert bool(torch.isfinite(y).all())
    mag = x.double().abs() @ wd.abs().t()
    assert bool(((y.double() - want).abs() <= (K + 3) * 2.0 ** -24 * mag + 2.0 ** -23 * want.abs()).all())


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_infinite_scale(M, N, K):
    """f32(0) * inf is NaN in the effective weight, so a channel with an infinite scale is NaN where
    any of its weights is 0, and an infinity of the sum's sign, or NaN, elsewhere."""
    g = torch.Generator(device="cuda").manual_seed(M + K)
    x = torch.rand(M, K, generator=g, device="cuda") + 0.5
    q = torch.randint(1, 128, (N, K), generator=g, device="cuda")
    s = torch.full((N,), 0.01, device="cuda")
    s[0], s[N // 2], s[N - 1] = INF, INF, INF
    q[0, 3] = 0
    q[N // 2, 5] = -1
    y = I.linear_w8a32(x, _packed(q, s))
    assert bool(torch.isnan(y[:, 0]).all()) and bool(torch.isnan(y[:, N // 2]).all())  # 0 * inf; inf - inf
    assert bool((y[:, N - 1] == INF).all())
    rest = torch.ones(N, dtype=torch.bool, device="cuda")
    rest[[0, N // 2, N - 1]] = False
    assert bool(torch.isfinite(y[:, rest]).all())


@pytest.mark.parametrize("M,N,K", SHAPES)
def test_non_finite_values(M, N, K):
    """Rows with one infinity, two of either sign, a NaN, only NaN, beside finite ones: NaN and
    infinity where float64 on the effective weights has them, the other rows' bits unchanged."""
    print(f"w8a32 non-finite M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    w8 = I.pack_linear_weight(torch.randn(N, K, generator=g, device="cuda"), weight_only=True)
    b = torch.randn(N, generator=g, device="cuda")
    plain = I.linear_w8a32(x, w8, b)
    xi = x.clone()
    at = torch.arange(M, device="cuda") % 7
    if M < 7:
        at[:4] = torch.arange(4, device="cuda")
    xi[at == 0, K - 1] = INF
    xi[at == 1, 2] = -INF
    xi[at == 1, K // 2] = INF
    xi[at == 2, K // 3] = float("nan")
    xi[at == 3] = float("nan")
    y = I.linear_w8a32(xi, w8, b)
    wd = (w8.q.double() * w8.s.double()[:, None]).t().contiguous()
    bad = at < 4
    want = xi[bad].double() @ wd + b.double()
    assert torch.equal(torch.isnan(y[bad]), torch.isnan(want))
    inf = torch.isinf(want)
    assert bool(inf.any()) and torch.equal(y[bad][inf].double(), want[inf])
    assert torch.equal(y[~bad], plain[~bad])


@pytest.mark.parametrize("M,N,K", [(256, 1024, 4096), (2048, 2048, 512)])
def test_a_batch_of_nan_costs_little_more(M, N, K):
    """A NaN in x decides its row, so its outputs need no second sum: such a batch takes about
    twice the time of a finite one (30 times when each output was summed again)."""
    w8 = I.pack_linear_weight(torch.randn(N, K, device="cuda"), weight_only=True)

    def us(x):
        best = 1e9
        for _ in range(8):
            e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            e0.record()
            for _ in range(8):
                I.linear_w8a32(x, w8)
            e1.record()
            e1.synchronize()
            best = min(best, e0.elapsed_time(e1) * 125)
        return best
    x = torch.randn(M, K, device="cuda")
    t = us(x), us(torch.full_like(x, float("nan")))
    assert t[1] < 6 * t[0] + 20, t


@pytest.mark.parametrize("scale", [2.0 ** -100, 2.0 ** -112, 2.0 ** -118, 2.0 ** -124])
@pytest.mark.parametrize("M,N,K", SHAPES)
def test_tiny_values(M, N, K, scale):
    """Activations whose bf16 pieces fall below bf16's last bit, in rows of their own (scales of up
    to 2^30 keep the outputs normal numbers), beside ordinary rows and rows of zeros: within the f32
    accumulation's bound, and no bit of the others changed."""
    print(f"w8a32 tiny M={M} N={N} K={K} scale={scale}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    x = torch.randn(M, K, generator=g, device="cuda")
    q = torch.randint(-127, 128, (N, K), generator=g, device="cuda")
    q[1] = 0  # an empty output channel
    s = torch.exp2(30 * torch.rand(N, generator=g, device="cuda"))
    w8 = _packed(q, s)
    plain = I.linear_w8a32(x, w8)
    rows = torch.arange(M, device="cuda") % 3
    x[rows == 1] *= scale
    x[rows == 2] = 0
    y = I.linear_w8a32(x, w8)
    wd = (q.double() * s.double()[:, None]).t().contiguous()
    tiny = x[rows == 1].double()
    want, mag = tiny @ wd, tiny.abs() @ wd.abs()
    # an f32 sum over the effective weights or scaled after it (one more rounding), and underflow:
    # half of f32's last bit, 2^-150, a product and sum
    bound = (K + 3) * 2.0 ** -24 * mag + 2.0 ** -23 * want.abs() + 2 * K * 2.0 ** -150
    err = (y[rows == 1].double() - want).abs()
    assert bool((err <= bound).all()), float((err / bound).max())
    # and as a whole as close as ordinary values come (about 4e-7): the lost bits are 2^-17 of 2^-118
    assert float(err.norm() / want.norm()) < 2e-6
    assert torch.equal(y[rows == 0], plain[rows == 0]) and not bool(y[rows == 2].any())


@pytest.mark.parametrize("M,N,K", SHAPES + [(17, 1, 16), (257, 2050, 320), (1030, 2055, 272), (16, 1024, 2048)])
@pytest.mark.parametrize("act", [I.ACT_NONE, I.ACT_RELU, I.ACT_GELU])
def test_bias_residual_and_activation(M, N, K, act):
    """act((y + bias) + residual) of the same y, in every kernel; y within the f32 bound of float64."""
    print(f"w8a32 epilogue M={M} N={N} K={K} act={act}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    w8 = I.pack_linear_weight(torch.randn(N, K, generator=g, device="cuda"), weight_only=True)
    b, r = torch.randn(N, generator=g, device="cuda"), torch.randn(M, N, generator=g, device="cuda")
    y = I.linear_w8a32(x, w8)
    wd = (w8.q.double() * w8.s.double()[:, None]).t().contiguous()
    want = x.double() @ wd
    bound = (K + 3) * 2.0 ** -24 * (x.double().abs() @ wd.abs()) + 2.0 ** -23 * want.abs()
    assert bool(((y.double() - want).abs() <= bound).all())
    got = I.linear_w8a32(x, w8, b, act, residual=r)
    pre = (y + b) + r
    if act == I.ACT_GELU:
        assert torch.allclose(got, torch.nn.functional.gelu(pre), rtol=1e-5, atol=1e-6)
    else:
        assert torch.equal(got, torch.relu(pre) if act == I.ACT_RELU else pre)


# more slices than meet at a time (8 of a 16 x 16 block, 2 of the larger), unequal and short last ones
@pytest.mark.parametrize("M,N,K", [(16, 40, 8208), (5, 300, 8240), (3, 100, 16384), (12, 700, 4112), (33, 200, 8208),
                                   (20, 64, 12304), (128, 3000, 1520), (64, 1000, 4176), (200, 1024, 2064)])
def test_slices_in_turn(M, N, K):
    """Without a workspace the slices of K run in turn in other blocks: the same bits."""
    print(f"w8a32 in turn M={M} N={N} K={K}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N + K)
    x = torch.randn(M, K, generator=g, device="cuda")
    w8 = I.pack_linear_weight(torch.randn(N, K, generator=g, device="cuda"), weight_only=True)
    b = torch.randn(N, generator=g, device="cuda")
    out = torch.empty(M, N, device="cuda")
    check(lib().bq_linear_w8a32(x.data_ptr(), w8.q.data_ptr(), M, N, K, w8.s.data_ptr(), b.data_ptr(), None, 0,
                                out.data_ptr(), torch.cuda.current_stream().cuda_stream))
    assert torch.equal(out, I.linear_w8a32(x, w8, b))
