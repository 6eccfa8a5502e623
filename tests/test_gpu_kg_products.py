"""The moment products of real sequences, mu^{ab} = <B_a T_m r | T_n B_b r>, at the
edges of the tiles (32 A of 2 x 2 waves), of a block of sixteen of K and of
the chunks, against the sequences formed in NumPy in 64 bits. A Chebyshev
recurrence of M steps carries at most about M^2 roundings of its precision's
unit u: 4 (M + 2)^2 u of the largest element."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def ring(n, seed):
    rng = np.random.default_rng(seed)
    D = np.zeros((n, n))
    k = np.arange(n)
    D[k, k] = rng.uniform(-1, 1, n)
    B = [np.zeros((n, n)) for _ in range(3)]
    if n > 2:
        t = rng.uniform(-1, 1, n)
        D[k, (k + 1) % n] = D[(k + 1) % n, k] = t
        for b in B:
            t = rng.uniform(-1, 1, n)
            b[k, (k + 1) % n], b[(k + 1) % n, k] = t, -t
    return D, B


def bsr(D, pattern):
    r, c = np.nonzero(pattern)
    return BSR.from_blocks(D.shape[0], 1, r, c, D[r, c].reshape(-1, 1, 1))


# rows x columns = K: one element, below a block, a block, ragged blocks, one and several chunks
@pytest.mark.parametrize("n,R", [(1, 1), (5, 3), (8, 2), (17, 1), (13, 5), (64, 1), (65, 1), (331, 3), (1200, 7)])
@pytest.mark.parametrize("M", [1, 2, 33, 64, 65, 96, 97, 129, 200])
def test_moment_products(n, R, M):
    D, B = ring(n, n)
    pattern = (D != 0) | np.eye(n, dtype=bool)
    a = 1.05 * max(np.abs(np.linalg.eigvalsh(D)).max(), 0.1)
    psi = np.random.default_rng(R).standard_normal((n, R))
    for prec, u in ((_lib.PREC_FP64, 2.0 ** -53), (_lib.PREC_FP32, 2.0 ** -24)):
        with _lib.Context(0) as ctx:
            ctx.upload_bsr(_lib.SLOT_H, bsr(D, pattern))
            for d in range(3):
                ctx.upload_bsr(_lib.SLOT_VX + d, bsr(B[d], pattern))
            ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.0, a)
            ctx.set_samples(n, R, _lib.SAMPLES_UPLOAD_REAL, data=psi)
            mu = np.asarray(ctx.dc_spectrum(M, with_moments=True, precision=prec)[2])

        def chain(x):
            out = [x, D @ x / a]
            while len(out) < M:
                out.append(2 * (D @ out[-1]) / a - out[-2])
            return np.stack([v.reshape(-1) for v in out[:M]])

        T = chain(psi).reshape(M, n, R)
        want = []
        for b in B:
            left = np.stack([(b @ t).reshape(-1) for t in T])
            want.append(left @ chain(b @ psi).T / (4 * a * a))
        want = np.stack(want)
        assert np.abs(mu.imag).max() == 0.0
        assert np.abs(mu.real - want).max() <= 4 * (M + 2) ** 2 * u * np.abs(want).max()
