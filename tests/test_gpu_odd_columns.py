"""The tiled GEMM's one-column-a-lane epilogue against its general path, bit for bit."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402
from borch_amd._lib import check, lib  # noqa: E402


# tiles of every configuration the rule picks, ragged in rows and columns: 64 x 64, 128 x 128 (both
# rings), 256 x 256, 128 x 256, 320 x 256, 128 x 32; columns one past and one short of a tile
@pytest.mark.parametrize("M,N,K", [(65, 33, 48), (100, 1, 272), (300, 65, 784), (1000, 1002, 528), (1000, 2999, 1568),
                                   (2100, 1999, 512), (4095, 4095, 512), (6304, 767, 272), (6300, 3071, 96),
                                   (16500, 31, 64)])
@pytest.mark.parametrize("act", [I.ACT_NONE, I.ACT_RELU, I.ACT_SILU, I.ACT_GELU])
def test_odd_columns(M, N, K, act):
    """The f32 output alone (one column a lane) equals the general path's (int32 output asked for
    too) bit for bit, with and without a residual, and so does an unaligned output of aligned
    width; nothing is written past the output."""
    print(f"odd columns M={M} N={N} K={K} act={act}", flush=True)
    g = torch.Generator(device="cuda").manual_seed(M + N)
    qa = torch.randint(-127, 128, (M, K), generator=g, device="cuda", dtype=torch.int8)
    qw = torch.randint(-127, 128, (N, K), generator=g, device="cuda", dtype=torch.int8)
    sa, sw, b = (torch.rand(n, generator=g, device="cuda") * 1e-2 for n in (M, N, N))
    r = torch.randn(M, N, generator=g, device="cuda")
    for res in (None, r):
        want, acc = I.gemm_i8(qa, qw, sa, sw, b, act, want_acc=True, residual=res)
        assert torch.equal(acc.double(), qa.double() @ qw.double().t())
        assert torch.equal(I.gemm_i8(qa, qw, sa, sw, b, act, residual=res), want)
        buf = torch.full((M * N + 256,), 3.0, device="cuda")
        check(lib().bq_gemm_i8(qa.data_ptr(), qw.data_ptr(), M, N, K, sa.data_ptr(), sw.data_ptr(), b.data_ptr(),
                               None if res is None else res.data_ptr(), act, buf.data_ptr() + 4, None, None, 0,
                               torch.cuda.current_stream().cuda_stream))
        assert torch.equal(buf[1:1 + M * N].view(M, N), want)
        assert float(buf[0]) == 3.0 and bool((buf[1 + M * N:] == 3.0).all())
