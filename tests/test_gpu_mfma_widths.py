"""The MFMA SpMM at every kind of width: fewer, exactly and more columns than
its tiles hold, odd real widths, two chunks, real and complex matrices, rows
without blocks; products and moments against the oracle (FP64) and the FP32
form against it."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def _hermitian(nbr, b, cplx, seed, hole=True):
    """Random Hermitian BSR with about seven blocks a row; block row nbr // 2
    (and its column) is empty."""
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(nbr), 3)
    j = (i + rng.integers(1, max(2, nbr), i.size)) % nbr
    if hole and nbr > 2:
        keep = (i != nbr // 2) & (j != nbr // 2)
        i, j = i[keep], j[keep]
    off = i != j
    i, j = i[off], j[off]
    v = rng.standard_normal((i.size, b, b))
    d = rng.standard_normal((nbr, b, b))
    if cplx:
        v = v + 1j * rng.standard_normal(v.shape)
        d = d + 1j * rng.standard_normal(d.shape)
    d = d + np.conj(np.swapaxes(d, 1, 2))
    k = np.arange(nbr)
    if hole and nbr > 2:
        k, d = np.delete(k, nbr // 2), np.delete(d, nbr // 2, 0)
    return BSR.from_blocks(nbr, b, np.concatenate([k, i, j]), np.concatenate([k, j, i]),
                           np.concatenate([d, v, np.conj(np.swapaxes(v, 1, 2))]))


def _vec(rows, R, cplx, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, R))
    return x + 1j * rng.standard_normal((rows, R)) if cplx else x


# real widths 1 .. 256 and complex ones 2 .. 512 around every tile count
REAL_R = [1, 7, 15, 16, 17, 24, 33, 50, 96, 100, 129, 200, 255, 256]
CPLX_R = [1, 4, 8, 10, 16, 17, 24, 25, 48, 50, 64, 75, 96, 100, 128, 129, 150, 192, 200, 256]


@pytest.mark.parametrize("nbr,b", [(1, 8), (23, 9), (40, 13), (9, 16)])
def test_products_at_every_width(oracle, nbr, b):
    H, C = _hermitian(nbr, b, False, 1), _hermitian(nbr, b, True, 2)
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        ctx.upload_bsr(_lib.SLOT_S, C)
        for slot, M, cv, widths in ((_lib.SLOT_H, H, False, REAL_R), (_lib.SLOT_H, H, True, CPLX_R),
                                    (_lib.SLOT_S, C, True, CPLX_R)):
            for R in widths:
                x = _vec(M.n_rows, R, cv, 3 + R)
                y, ref = ctx.bsr_mult(slot, x), oracle.bsr_mult(M, x)
                # a row sums at most 7 b terms of size <= 20: 7 16 20 2^-52 << 1e-11
                assert np.max(np.abs(y - ref)) <= 1e-11, (slot, cv, R)


@pytest.mark.parametrize("b,cplx,R,kind", [
    (13, False, 7, "real"), (13, False, 16, "real"), (9, False, 50, "real"), (13, False, 10, "phase"),
    (13, False, 24, "phase"), (9, False, 75, "phase"), (13, False, 129, "phase"), (9, True, 1, "phase"),
    (9, True, 16, "phase"), (13, True, 20, "phase"), (13, True, 64, "phase"), (9, True, 128, "phase")])
@pytest.mark.parametrize("doubling", [_lib.DOUBLING_ON, _lib.DOUBLING_OFF])
def test_moments_at_every_width(oracle, b, cplx, R, kind, doubling):
    H = _hermitian(60, b, cplx, 5)
    a = 1.05 * np.abs(np.linalg.eigvalsh(H.to_dense())).max()
    rng = np.random.default_rng(6)
    psi = (rng.choice([-1.0, 1.0], (H.n_rows, R)) if kind == "real"
           else np.exp(2j * np.pi * rng.random((H.n_rows, R)))) / np.sqrt(H.n_rows)
    M = 24
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.1, a)
        ctx.set_samples(H.n_rows, R, _lib.SAMPLES_UPLOAD_REAL if kind == "real" else _lib.SAMPLES_UPLOAD_COMPLEX,
                        data=psi)
        mu, cols = ctx.kpm_moments(M, doubling=doubling, per_column=True)
        mu32 = ctx.kpm_moments(M, precision=_lib.PREC_FP32, doubling=doubling)
        again = ctx.kpm_moments(M, doubling=doubling)
    op = oracle.Operator(oracle.FORM_ORTHOGONAL, H, 0.1, a)
    ref = op.moments(psi, M, doubling=doubling == _lib.DOUBLING_ON)
    assert np.max(np.abs(mu - ref)) <= 1e-12
    assert np.max(np.abs(cols.mean(axis=1) - ref)) <= 1e-12
    assert np.array_equal(mu, again)
    # single precision over 24 steps of a bounded recurrence
    assert np.max(np.abs(mu32 - ref)) <= 2e-5
