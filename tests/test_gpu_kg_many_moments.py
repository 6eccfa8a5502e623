"""Moment products of real sequences with few chunks of K: exactly, and at a
rate near that of many chunks.

H is diagonal with eigenvalues of cosines 0, 1/2 and 1, so every Chebyshev vector
holds multiples of 1/2 only, and with small integers in the samples and velocity
factors every product and sum is exact in FP32 sequences and FP64 sums: the
moments of NumPy are met bit for bit, whatever the order of the sums."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def operators(n, rng):
    """(H, velocity factors) of a ring on one pattern, and their dense forms."""
    k = np.arange(n)
    rows, cols = np.concatenate([k, k, (k + 1) % n]), np.concatenate([k, (k + 1) % n, k])
    h = rng.choice([-1.0, -0.5, 0.0, 0.5, 1.0], n)

    def bsr(d, t, sign):
        return BSR.from_blocks(n, 1, rows, cols, np.concatenate([d, t, sign * t]).reshape(-1, 1, 1))

    ts = [rng.integers(-2, 3, n).astype(float) for _ in range(3)]
    return h, ts, bsr(h, np.zeros(n), 1.0), [bsr(np.zeros(n), t, -1.0) for t in ts]


def apply_factor(t, x):
    # B[k, k + 1] = t[k], B[k + 1, k] = -t[k]
    y = t[:, None] * np.roll(x, -1, 0)
    y -= np.roll(t[:, None] * x, 1, 0)
    return y


def context(n, R, H, V, psi):
    ctx = _lib.Context(0)
    ctx.upload_bsr(_lib.SLOT_H, H)
    for d in range(3):
        ctx.upload_bsr(_lib.SLOT_VX + d, V[d])
    ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.0, 1.0)
    ctx.set_samples(n, R, _lib.SAMPLES_UPLOAD_REAL, data=psi)
    return ctx


# K = n R: one chunk, a few, all that the tiles leave; ragged last blocks
@pytest.mark.parametrize("n,R", [(37, 1), (331, 3), (1024, 1)])
@pytest.mark.parametrize("M", [33, 200, 640, 1030, 1100, 1500, 2050])
@pytest.mark.parametrize("formulation", [0, 1])
def test_moments_are_exact(n, R, M, formulation):
    rng = np.random.default_rng(n + M)
    h, ts, H, V = operators(n, rng)
    psi = rng.integers(-3, 4, (n, R)).astype(float)
    cheb = [np.ones(n), h]
    while len(cheb) < M:
        cheb.append(2.0 * h * cheb[-1] - cheb[-2])
    T = np.stack(cheb[:M])[:, :, None]
    left = [np.stack([apply_factor(t, x).reshape(-1) for x in T * psi]) for t in ts]
    right = [(T * apply_factor(t, psi)).reshape(M, -1) for t in ts]
    pairs = [(0, 0), (0, 1), (0, 2), (1, 1), (1, 2), (2, 2)] if formulation else [(0, 0), (1, 1), (2, 2)]
    want = np.stack([left[a] @ right[b].T for a, b in pairs]) / 4.0
    for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
        print("case: exact moments", n, R, M, formulation, prec, flush=True)
        with context(n, R, H, V, psi) as ctx:
            mu = np.asarray(ctx.dc_spectrum(M, formulation, with_moments=True, precision=prec)[2])
        assert np.abs(mu.imag).max() == 0.0
        assert np.array_equal(mu.real, want)


def test_rate_does_not_fall_with_the_moments():
    """1,500 moments leave each product one to eight chunks of K; their rate is at
    least half of that of 512 moments (sixteen chunks)."""
    def rate(M, n, R):
        rng = np.random.default_rng(M)
        _, _, H, V = operators(n, rng)
        with context(n, R, H, V, rng.integers(-3, 4, (n, R)).astype(float)) as ctx:
            best = 0.0
            for _ in range(4):
                ctx.set_profiling(True)
                ctx.dc_spectrum(M)
                s = ctx.kernel_stats(_lib.KCLASS_KG_GEMM)
                best = max(best, s["flops"] / s["avg_ms"])
        return best

    assert rate(1500, 4096, 16) >= 0.5 * rate(512, 8192, 16)


@pytest.mark.parametrize("formulation", [0, 1])
@pytest.mark.parametrize("limit", ["0", "100000", "3000000"])
def test_moments_without_room_for_the_parts(formulation, limit, monkeypatch):
    """Fewer chunks of K, or one product at a time, give the same exact moments."""
    n, R, M = 1024, 1, 200
    rng = np.random.default_rng(8)
    h, ts, H, V = operators(n, rng)
    psi = rng.integers(-3, 4, (n, R)).astype(float)
    with context(n, R, H, V, psi) as ctx:
        want = ctx.dc_spectrum(M, formulation, with_moments=True)[2]
        full = ctx.mem_info()[0]
    monkeypatch.setenv("RG_STORE_MAX", limit)
    with context(n, R, H, V, psi) as ctx:
        for prec in (_lib.PREC_FP64, _lib.PREC_FP32):
            assert np.array_equal(ctx.dc_spectrum(M, formulation, with_moments=True, precision=prec)[2], want)
        # sixteen chunks of three or six products, 256 x 256 each, take 25 MB or 50
        assert ctx.mem_info()[0] - full > 16 * (1 << 20)
