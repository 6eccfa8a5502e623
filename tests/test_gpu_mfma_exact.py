"""Every shape of the MFMA SpMM's moment steps in exact arithmetic: blocks of -1,
0, 1 (and i), samples of +-1 (and +-i) and a window of 64 keep three steps of the
recurrence within 24 bits and their dots within 53, so the per-column moments of
both precisions equal the ones formed from the oracle's products, bit for bit
and in any order of the sums. The widths stand on both sides of every tile
count, access size and column split of the dispatch, in operators of fewer and
of more block rows than the split asks for."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu

REAL_R = [1, 15, 16, 17, 18, 30, 31, 32, 33, 34, 36, 64, 65, 66, 68, 96, 98, 100, 128, 129, 130, 132, 192, 194, 196, 200, 255, 256]
CPLX_R = [1, 2, 8, 9, 16, 17, 24, 25, 32, 33, 34, 48, 49, 64, 65, 66, 75, 96, 97, 98, 100, 128, 129, 130, 150, 192, 200, 255,
          256]
WINDOW = 64.0


def integer_hermitian(nbr, b, cplx, seed):
    rng = np.random.default_rng(seed)
    i = np.repeat(np.arange(nbr), 2)
    j = (i + rng.integers(1, max(2, nbr), i.size)) % nbr
    i, j = i[i != j], j[i != j]

    def ints(n):
        v = rng.integers(-1, 2, (n, b, b)).astype(float)
        return v + 1j * rng.integers(-1, 2, (n, b, b)) if cplx else v

    v, d = ints(i.size), ints(nbr)
    d = np.triu(d, 1)
    d = d + np.conj(np.swapaxes(d, 1, 2))
    k = np.arange(nbr)
    return BSR.from_blocks(nbr, b, np.concatenate([k, i, j]), np.concatenate([k, j, i]),
                           np.concatenate([d, v, np.conj(np.swapaxes(v, 1, 2))]))


def exact_columns(oracle, H, psi, M, doubled):
    """Moments of every column from the oracle's products (all exact here)."""
    def dot(x, y):
        return np.sum(np.conj(x) * y, axis=0)

    t = [psi, oracle.bsr_mult(H, psi) / WINDOW]
    while len(t) < (M // 2 + 1 if doubled else M):
        t.append(2.0 * oracle.bsr_mult(H, t[-1]) / WINDOW - t[-2])
    for m, v in enumerate(t):  # whole multiples of 64^-m below 2^24 of them
        n = np.stack([v.real, v.imag]) * WINDOW ** m
        assert np.array_equal(n, np.rint(n)) and np.abs(n).max() < 2 ** 24
    if not doubled:
        return np.stack([dot(t[0], v) for v in t[:M]])
    mu = [dot(t[0], t[0]), dot(t[0], t[1])]
    while len(mu) < M:
        n = len(mu) // 2
        mu.append(2.0 * (dot(t[n], t[n]) if len(mu) % 2 == 0 else dot(t[n + 1], t[n])) - mu[len(mu) % 2])
    return np.stack(mu[:M])


def check(oracle, nbr, b, cplx, real_R, cplx_R):
    H = integer_hermitian(nbr, b, cplx, nbr + b)
    rng = np.random.default_rng(b)
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.0, WINDOW)
        for R, cv in [(r, False) for r in real_R if not cplx] + [(r, True) for r in cplx_R]:
            psi = rng.choice([1, -1, 1j, -1j], (H.n_rows, R)) if cv else rng.choice([-1.0, 1.0], (H.n_rows, R))
            ctx.set_samples(H.n_rows, R, _lib.SAMPLES_UPLOAD_COMPLEX if cv else _lib.SAMPLES_UPLOAD_REAL, data=psi)
            for M, doubling in ((6, _lib.DOUBLING_ON), (4, _lib.DOUBLING_OFF)):
                want = exact_columns(oracle, H, psi, M, doubling == _lib.DOUBLING_ON)
                for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
                    cols = ctx.kpm_moments(M, precision=prec, doubling=doubling, per_column=True)[1]
                    assert np.array_equal(cols, want), (R, cv, M, prec)


@pytest.mark.parametrize("b", [8, 9, 13, 16])
@pytest.mark.parametrize("cplx", [False, True])
def test_few_block_rows(oracle, b, cplx):
    check(oracle, 37, b, cplx, REAL_R, CPLX_R)


@pytest.mark.parametrize("cplx", [False, True])
def test_many_block_rows(oracle, cplx):
    """1,700 block rows: the shapes that few block rows split over more waves."""
    check(oracle, 1700, 9, cplx, [32, 64, 128, 256], [16, 32, 64, 128, 256])
