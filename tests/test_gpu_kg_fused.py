"""The one-launch-a-moment sequences of the conductivity spectrum against the
launches one by one (profiling, and a velocity on another pattern, ask for
those): moments and spectra bit for bit, over widths (whole 16-byte pieces,
odd), both sample kinds and precisions, ragged rows, few moments."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def _operators(n, seed):
    """Ragged symmetric H and three antisymmetric factors on its pattern."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(n), rng.integers(0, 6, n))
    j = rng.integers(0, n, i.size)
    keep = i != j
    key = np.unique(np.minimum(i, j)[keep] * n + np.maximum(i, j)[keep])
    i, j = key // n, key % n
    k = np.arange(n)

    def bsr(d, v, sign):
        return BSR.from_blocks(n, 1, np.concatenate([k, i, j]), np.concatenate([k, j, i]),
                               np.concatenate([d, v, sign * v]).reshape(-1, 1, 1))

    H = bsr(rng.uniform(-1, 1, n), rng.uniform(-1, 1, i.size), 1.0)
    return H, [bsr(np.zeros(n), rng.uniform(-1, 1, i.size), -1.0) for _ in range(3)]


def _spectrum(H, V, psi, M, formulation, prec, apart):
    a = 1.1 * float(np.max(np.bincount(H.block_rows(), np.abs(H.values.reshape(-1)), H.n_rows))) + 0.1
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        for d in range(3):
            ctx.upload_bsr(_lib.SLOT_VX + d, V[d])
        ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.05, a)
        ctx.set_samples(H.n_rows, psi.shape[1],
                        _lib.SAMPLES_UPLOAD_COMPLEX if np.iscomplexobj(psi) else _lib.SAMPLES_UPLOAD_REAL, data=psi)
        if apart:
            ctx.set_profiling(True)
        return ctx.dc_spectrum(M, formulation, with_moments=True, precision=prec)


@pytest.mark.parametrize("n,M", [(1, 1), (5, 2), (301, 3), (700, 24)])
@pytest.mark.parametrize("R,cplx", [(1, True), (2, False), (7, False), (10, False), (12, True), (32, True)])
@pytest.mark.parametrize("formulation", [0, 1])
def test_fused_sequences_equal_single_launches(n, M, R, cplx, formulation):
    H, V = _operators(n, n)
    rng = np.random.default_rng(R)
    psi = rng.standard_normal((n, R)) + (1j * rng.standard_normal((n, R)) if cplx else 0.0)
    for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
        one = _spectrum(H, V, psi, M, formulation, prec, False)
        apart = _spectrum(H, V, psi, M, formulation, prec, True)
        for x, y in zip(one, apart):
            assert np.array_equal(x, y)


def test_another_velocity_pattern_is_not_fused():
    H, V = _operators(400, 9)
    far = [(r, c) for r, c in ((0, 399), (3, 250), (17, 333)) if c not in H.col_ind[H.row_ptr[r]:H.row_ptr[r + 1]]]
    assert far
    r, c = far[0]
    rows = np.concatenate([V[2].block_rows(), [r, c]])
    cols = np.concatenate([V[2].col_ind, [c, r]])
    W = BSR.from_blocks(400, 1, rows, cols, np.concatenate([V[2].values, [[[0.3]], [[-0.3]]]]))
    # same entry count as H, another place: one entry pair dropped elsewhere
    first = int(np.flatnonzero(W.block_rows() != W.col_ind)[0])
    p, q = int(W.block_rows()[first]), int(W.col_ind[first])
    keep = ~(((W.block_rows() == p) & (W.col_ind == q)) | ((W.block_rows() == q) & (W.col_ind == p)))
    W = BSR.from_blocks(400, 1, W.block_rows()[keep], W.col_ind[keep], W.values[keep])
    assert W.nnzb == H.nnzb and not np.array_equal(W.col_ind, H.col_ind)
    psi = np.random.default_rng(1).standard_normal((400, 4))
    one = _spectrum(H, [V[0], V[1], W], psi, 12, 0, _lib.PREC_FP64, False)
    apart = _spectrum(H, [V[0], V[1], W], psi, 12, 0, _lib.PREC_FP64, True)
    for x, y in zip(one, apart):
        assert np.array_equal(x, y)
