"""The weight-only Linear at the ends of its size range, in every kernel: empty products."""
from __future__ import annotations

import pytest
import torch

pytestmark = pytest.mark.gpu

from borch_amd import int8 as I  # noqa: E402
from borch_amd._lib import check, lib  # noqa: E402

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
