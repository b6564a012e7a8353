"""The weight-only Linear's bf16-MFMA kernels (bq_linear_w8a32_ws) at the edges of their tiles
and slices: outputs within the f32-accumulation bound of the float64 result on the same
effective weights, the sliced sums' bits independent of the workspace, and non-finite
activations as f32 arithmetic gives them."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402
from borch_amd._lib import check, lib  # noqa: E402


def _case(M, N, K, seed=0):
    g = torch.Generator(device="cuda").manual_seed(seed)
    x = torch.randn(M, K, generator=g, device="cuda") * torch.exp(2 * torch.randn(M, 1, generator=g, device="cuda"))
    w8 = I.pack_linear_weight(torch.randn(N, K, generator=g, device="cuda"), weight_only=True)
    return x, w8, torch.randn(N, generator=g, device="cuda")


def _bounded(y, x, w8, b, K, act=None):
    """Within (K + 2) 2^-24 sum |x w| + 2^-24 |y| (one rounding a product and a sum, Higham's
    gamma_K) plus the bias addition's half ulp, of the float64 result; the bf16 kernels scale
    the sum where the bound's weights are f32(q) * s, one more rounding of 2^-24 sum |x w|."""
    K0 = x.shape[1]
    w = w8.q.double()[:, :K0] * w8.s.double()[:, None]
    ref = x.double() @ w.t()
    bound = (K + 3) * 2.0 ** -24 * (x.double().abs() @ w.abs().t()) + 2.0 ** -23 * (ref.abs() + b.double().abs())
    err = (y.double() - (ref + b.double())).abs()
    assert bool((err <= bound).all()), f"max err / bound {float((err / bound).max())}"


# rows: the f32-MFMA kernel's range and its edge, each K-split tile's remainders, the tiled
# kernel's 64 x 64 and 64 x 128 workgroups; columns odd, below one tile and past one; K one 16-value piece, a
# piece past a chunk, and slices of unequal length
@pytest.mark.parametrize("M,N,K", [(5, 17, 16), (16, 65, 1040), (13, 129, 2064), (16, 4096, 2048), (16, 63, 8208),
                                   (6, 4100, 4096), (17, 1, 80), (31, 130, 4112), (32, 4096, 1024), (33, 127, 528),
                                   (65, 4097, 2064), (200, 3000, 784), (257, 2050, 1040), (1030, 2055, 272),
                                   (2050, 2050, 144), (4097, 513, 96), (6304, 768, 80)])
def test_edges(M, N, K):
    print(f"w8a32 edges M={M} N={N} K={K}", flush=True)
    x, w8, b = _case(M, N, K, M + N + K)
    _bounded(I.linear_w8a32(x, w8, b), x, w8, b, K)


@pytest.mark.parametrize("M,N,K", [(16, 4096, 4096), (8, 300, 4112), (20, 768, 3072), (64, 1024, 1024), (40, 4100, 2064),
                                   (128, 500, 4096)])
def test_sliced_sums_do_not_depend_on_the_workspace(M, N, K):
    """Slices on their own workgroups (a workspace) or in turn in one (none): the same bits, the
    counters zero again after every call, also from a replayed graph."""
    print(f"w8a32 slices M={M} N={N} K={K}", flush=True)
    x, w8, b = _case(M, N, K, 1)
    ws = torch.zeros(int(lib().bq_gemm_ws_bytes()), dtype=torch.uint8, device="cuda")
    outs = [torch.empty(M, N, device="cuda") for _ in range(3)]

    def call(out, w, size):
        check(lib().bq_linear_w8a32_ws(x.data_ptr(), w8.q.data_ptr(), M, N, K, w8.s.data_ptr(), b.data_ptr(), None, 0,
                                       out.data_ptr(), w, size, torch.cuda.current_stream().cuda_stream))
    call(outs[0], None, 0)
    for _ in range(3):
        call(outs[1], ws.data_ptr(), ws.numel())
        assert torch.equal(outs[0], outs[1]) and int(ws[:4096].count_nonzero()) == 0
    s = torch.cuda.Stream()
    with torch.cuda.stream(s):
        call(outs[2], ws.data_ptr(), ws.numel())
        g = torch.cuda.CUDAGraph()
        with torch.cuda.graph(g, stream=s):
            call(outs[2], ws.data_ptr(), ws.numel())
    torch.cuda.synchronize()
    for _ in range(3):
        outs[2].zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(outs[0], outs[2])


@pytest.mark.parametrize("M", [6, 16, 40, 600])
def test_non_finite_rows(M):
    """Rows with an infinity, a NaN, or a value that rounds to a bf16 infinity: as f32 products
    and sums give them (0 * inf and inf - inf are NaN); the other rows are untouched."""
    print(f"w8a32 non-finite M={M}", flush=True)
    N, K = 2048, 2064
    x, w8, b = _case(M, N, K, 2)
    plain = I.linear_w8a32(x, w8, b)
    xi = x.clone()
    xi[0, 3], xi[1, 5], xi[2, 7], xi[3, 9], xi[4, 1], xi[4, 2] = (float("inf"), float("-inf"), float("nan"), 3.4e38,
                                                              float("inf"), float("inf"))
    xi[3] *= 2.0 ** -20
    xi[3, 9] = 3.4e38
    y = I.linear_w8a32(xi, w8, b)
    q = w8.q.double()[:, :K]
    for r, cols in ((0, [3]), (1, [5]), (2, [7]), (4, [1, 2])):
        want = (xi[r, cols].double()[None] * q[:, cols]).sum(1)  # the non-finite products decide the row
        fin = torch.isfinite(want)
        assert not bool(fin.any())
        assert torch.equal(torch.isnan(y[r]), torch.isnan(want))
        ok = ~torch.isnan(want)
        assert torch.equal(y[r][ok].double(), want[ok])
    sums = (xi[3].double() @ q.t())
    want = (sums * w8.s.double() + b.double()).float()  # infinite past f32's range only, whatever the sum before its scale
    assert bool((sums.abs() > 3.5e38)[torch.isfinite(want)].any())
    assert torch.allclose(y[3], want, rtol=1e-5)
    assert torch.equal(y[5:], plain[5:])
