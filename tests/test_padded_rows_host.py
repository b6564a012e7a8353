"""Size limits of the padding passes (bq_quantize_rows_padded, bq_pad_rows_f32), checked on the host
before any launch."""
import pytest

from borch_amd import _lib


@pytest.mark.parametrize("Kp", [0x7ffffff0, 0x7ffffc00, 0x7ffff010])
def test_rows_whose_next_index_leaves_an_int_are_refused(Kp):
    """A thread steps 1024 values through a row: past Kp = 2^31 - 4096 that index would wrap, and its
    loop over the row would not end. The pointers are never read."""
    lib = _lib.lib()
    assert lib.bq_quantize_rows_padded(16, 1, Kp - 8, Kp, 16, 16, None) == _lib.BQ_ERR_ARG
    assert "too large" in _lib.last_error()
    assert lib.bq_pad_rows_f32(16, 1, Kp - 8, Kp, 16, None) == _lib.BQ_ERR_ARG
    assert "too large" in _lib.last_error()
