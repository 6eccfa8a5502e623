"""The one-workgroup-per-column moment loop of small scalar operators against
the launched kernels (RG_GRAPH=0 asks for them) and the oracle: row counts
around a wave, a workgroup and two and four rows a thread, entries in registers
and read every step, empty and long rows, both precisions, real and complex
samples, step counts around its ring of sums and its longest launch."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def _matrix(n, per, seed):
    """Symmetric, about `per` off-diagonal entries a row; row 1 is empty and
    row 2 has twice as many when there is room."""
    rng = np.random.default_rng(seed)
    i = np.concatenate([np.repeat(np.arange(n), max(1, per // 2)), np.full(per, min(2, n - 1))])
    j = rng.integers(0, n, i.size)
    keep = (i != j) & (i != 1) & (j != 1)
    i, j = i[keep], j[keep]
    key = np.unique(np.minimum(i, j) * n + np.maximum(i, j))
    i, j = key // n, key % n
    v = rng.uniform(-1.0, 1.0, i.size)
    d = np.delete(np.arange(n), [1] if n > 1 else [])
    return BSR.from_blocks(n, 1, np.concatenate([d, i, j]), np.concatenate([d, j, i]),
                           np.concatenate([rng.uniform(-1, 1, d.size), v, v]).reshape(-1, 1, 1))


def _chain(n, seed):
    """A ring with onsite disorder: three entries a row."""
    rng = np.random.default_rng(seed)
    k = np.arange(n)
    return BSR.from_blocks(n, 1, np.concatenate([k, k, (k + 1) % n]), np.concatenate([k, (k + 1) % n, k]),
                           np.concatenate([rng.uniform(-1, 1, n), np.ones(2 * n)]).reshape(-1, 1, 1))


def _moments(monkeypatch, onchip, H, a, psi, M, prec, noalloc=False):
    if onchip:
        monkeypatch.delenv("RG_GRAPH", raising=False)
    else:
        monkeypatch.setenv("RG_GRAPH", "0")
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.05, a)
        ctx.set_samples(H.n_rows, psi.shape[1],
                        _lib.SAMPLES_UPLOAD_COMPLEX if np.iscomplexobj(psi) else _lib.SAMPLES_UPLOAD_REAL, data=psi)
        mu, cols = ctx.kpm_moments(M, prec, per_column=True)
        if noalloc:
            m2, c2 = ctx.kpm_moments_noalloc(M, prec, per_column=True)
            assert np.array_equal(mu, m2) and np.array_equal(cols, c2)
    return mu, cols


CASES = [("chain", 3, 0), ("chain", 64, 0), ("chain", 1000, 0), ("chain", 1025, 0), ("chain", 2049, 0),
         ("chain", 4096, 0), ("chain", 8192, 0), ("chain", 8193, 0), ("random", 5, 3), ("random", 320, 10), ("random", 1024, 6), ("random", 700, 28),
         ("random", 1500, 8), ("random", 3001, 5)]


@pytest.mark.parametrize("kind,n,per", CASES)
@pytest.mark.parametrize("R,cplx", [(1, True), (7, False), (16, True)])
def test_matches_launched_kernels_and_oracle(monkeypatch, oracle, kind, n, per, R, cplx):
    H = _chain(n, n) if kind == "chain" else _matrix(n, per, n)
    a = 1.1 * float(np.max(np.bincount(H.block_rows(), np.abs(H.values.reshape(-1)), n))) + 0.1
    rng = np.random.default_rng(n + R)
    psi = rng.standard_normal((n, R)) + (1j * rng.standard_normal((n, R)) if cplx else 0.0)
    psi /= np.linalg.norm(psi, axis=0)
    M = 141  # 70 steps: past one ring of 64
    for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
        mu, cols = _moments(monkeypatch, True, H, a, psi, M, prec, noalloc=True)
        mu0, cols0 = _moments(monkeypatch, False, H, a, psi, M, prec)
        # the vectors are the same bit for bit; FP64 sums of at most 8193 terms
        # of size <= 1 in another order
        assert np.max(np.abs(cols - cols0)) <= 4e-13
        assert np.max(np.abs(mu - mu0)) <= 4e-13
        if prec == _lib.PREC_FP64:
            ref = oracle.Operator(oracle.FORM_ORTHOGONAL, H, 0.05, a).moments(psi, M)
            assert np.max(np.abs(mu - ref)) <= 1e-12


@pytest.mark.parametrize("M", [1, 2, 3, 4, 5, 129, 130, 131, 132, 16386, 16500])
def test_step_counts(monkeypatch, M):
    H = _chain(100, 5)
    psi = np.random.default_rng(1).choice([-1.0, 1.0], (100, 2)) / 10.0
    mu, cols = _moments(monkeypatch, True, H, 3.3, psi, M, _lib.PREC_FP64, noalloc=True)
    mu0, cols0 = _moments(monkeypatch, False, H, 3.3, psi, M, _lib.PREC_FP64)
    assert np.max(np.abs(cols - cols0)) <= 1e-13
