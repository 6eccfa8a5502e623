"""The overlap factor on patches larger than the one-wave kernel's, by size
around the 16, 64 and block-table edges, ragged rows included: the symmetric
products against the eigendecomposition, and an overlap that is not symmetric
(it keeps the general products) against a matrix square root."""
import numpy as np
import pytest
from scipy.linalg import inv, sqrtm

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def _ring(nbr, b, reach, seed, drop=0.0, skew=0.0):
    """S = I + random symmetric couplings of every block to its `reach`
    neighbours on either side of a ring (spectrum inside [0.4, 1.6])."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(nbr), reach)
    j = (i + np.tile(np.arange(1, reach + 1), nbr)) % nbr
    keep = rng.random(i.size) >= drop
    i, j = i[keep], j[keep]
    v = rng.uniform(-1.0, 1.0, (i.size, b, b)) * (0.3 / (2 * reach * b))
    back = np.swapaxes(v, 1, 2) * (1.0 + skew)
    k = np.arange(nbr)
    return BSR.from_blocks(nbr, b, np.concatenate([k, i, j]), np.concatenate([k, j, i]),
                           np.concatenate([np.broadcast_to(np.eye(b), (nbr, b, b)), v, back]))


def _rows(S, f):
    """Block row i of f(S[C_i, C_i]) on S's pattern."""
    b, D = S.block_dim, S.to_dense()
    out = np.zeros_like(S.values)
    for r in range(S.n_block_rows):
        s = slice(int(S.row_ptr[r]), int(S.row_ptr[r + 1]))
        c = S.col_ind[s]
        idx = (c[:, None] * b + np.arange(b)).reshape(-1)
        me = int(np.flatnonzero(c == r)[0])
        out[s] = np.swapaxes(f(D[np.ix_(idx, idx)])[me * b:(me + 1) * b].reshape(b, -1, b), 0, 1)
    return out


def _eigh(A):
    w, U = np.linalg.eigh(A)
    return (U / np.sqrt(w)) @ U.T


def _factor(S):
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_S, S)
        it, res = ctx.isqrt_patches()
        Z, ZH = ctx.download_bsr(_lib.SLOT_Z), ctx.download_bsr(_lib.SLOT_ZH)
    assert 0 < it < 20 and res < 1e-12
    assert np.array_equal(Z.conj_transpose().values, ZH.values)
    return Z.values


@pytest.mark.parametrize("nbr,b,reach,drop", [
    (9, 6, 1, 0.0),    # 18: one tile of 32
    (9, 16, 1, 0.0),   # 48
    (11, 16, 2, 0.0),  # 80
    (20, 13, 2, 0.0),  # 65, just past a tile
    (37, 13, 8, 0.0),  # 221
    (40, 13, 8, 0.3),  # ragged
    (80, 1, 33, 0.0),  # 67 blocks: past the block table
    (30, 16, 9, 0.2),  # up to 304
])
def test_symmetric_patches(nbr, b, reach, drop):
    S = _ring(nbr, b, reach, 7 + nbr, drop)
    # Newton-Schulz to ||I - Z Y||_F < 1e-12 with condition numbers below 4
    assert np.max(np.abs(_factor(S) - _rows(S, _eigh))) < 1e-11


def test_unsymmetric_overlap_keeps_the_general_products():
    S = _ring(14, 8, 2, 3, skew=0.05)
    assert np.max(np.abs(_factor(S) - _rows(S, lambda A: inv(sqrtm(A).real)))) < 1e-11


def test_symmetric_up_to_rounding():
    S = _ring(14, 8, 2, 3)
    T = BSR(S.n_block_rows, S.block_dim, S.row_ptr, S.col_ind, S.values.copy())
    T.values[1::3] *= 1.0 + 2.0 ** -52
    assert np.max(np.abs(_factor(T) - _rows(S, _eigh))) < 1e-11
