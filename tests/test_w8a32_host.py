"""Host side of the weight-only Linear's C entries, without a GPU: what a call does before its
launch. Each runs in a process of its own that sees no device, so that a launch returns an error
and an abort is seen as one."""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parent.parent

_CALL = """
import ctypes, sys
from borch_amd._lib import lib
buf = ctypes.create_string_buffer(1 << 16)
at = (ctypes.addressof(buf) + 15) // 16 * 16
M, N, K = (int(v) for v in sys.argv[1:])
rc = [lib().bq_linear_w8a32(at, at, M, N, K, at, at, None, 0, at, None),
      lib().bq_linear_w8a32_ws(at, at, M, N, K, at, at, None, 0, at, None, 0, None)]
print("returned", *rc)
"""


@pytest.mark.parametrize("M,N", [(2, 16), (8, 16), (17, 1), (32, 16), (300, 300), (2048, 2048)])
def test_an_empty_product_returns(M, N):
    """K = 0 (the outputs are act(bias + residual)) reaches the launch: no shape rule divides by its
    count of K chunks."""
    env = dict(os.environ, HIP_VISIBLE_DEVICES="-1", ROCR_VISIBLE_DEVICES="-1", PYTHONPATH=str(ROOT))
    r = subprocess.run([sys.executable, "-c", _CALL, str(M), str(N), "0"], env=env, capture_output=True, text=True,
                       timeout=120)
    assert r.returncode == 0 and r.stdout.startswith("returned"), (r.returncode, r.stdout, r.stderr[-300:])
