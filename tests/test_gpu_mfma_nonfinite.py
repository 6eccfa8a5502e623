"""The MFMA SpMM with infinities and NaN in the vectors: a block row reads the
X rows of its own block columns only, so every other output is what it is
without them (the last K step of a row whose 7 or 9 blocks of 9 or 13 columns
do not fill steps of four reads past the row's panel)."""
import numpy as np
import pytest

from rsatb_amd import _lib
from test_gpu_mfma_widths import _hermitian, _vec

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("b", [8, 9, 11, 13, 14])
@pytest.mark.parametrize("cplx", [False, True])
@pytest.mark.parametrize("bad", [np.inf, np.nan])
def test_other_rows_keep_their_values(b, cplx, bad):
    H = _hermitian(31, b, cplx, b)
    dense_pattern = np.zeros((31, 31), bool)
    dense_pattern[H.block_rows(), H.col_ind] = True
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        for cv, widths in ((False, [] if cplx else [1, 16, 20, 32, 50, 64, 128, 256]),
                           (True, [1, 8, 10, 20, 32, 64, 75, 128, 150, 256])):
            for R in widths:
                x = _vec(H.n_rows, R, cv, R)
                clean = ctx.bsr_mult(_lib.SLOT_H, x)
                for blk in (0, 3, 7, 12, 21, 30):
                    y = x.copy()
                    y[blk * b] = bad  # a block's first column is what the next row's panel starts with
                    got = ctx.bsr_mult(_lib.SLOT_H, y).reshape(31, b, R)
                    touched = dense_pattern[:, blk]
                    ref = clean.reshape(31, b, R)
                    assert np.array_equal(got[~touched], ref[~touched]), (cv, R, blk)
                    assert not np.any(np.isfinite(got[touched])), (cv, R, blk)
