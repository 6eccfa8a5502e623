"""Device memory that a context holds beside what a call needs: given back, bounded,
or done without when there is no room."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu

MB = 1 << 20


def ring_blocks(n, b, width, seed):
    """Symmetric block rows of the diagonal and `width` neighbours a side."""
    rng = np.random.default_rng(seed)
    k = np.arange(n)
    d = rng.standard_normal((n, b, b))
    rows, cols, vals = [k], [k], [d + np.swapaxes(d, 1, 2)]
    for s in range(1, width + 1):
        v = rng.standard_normal((n, b, b))
        rows += [k, (k + s) % n]
        cols += [(k + s) % n, k]
        vals += [v, np.swapaxes(v, 1, 2)]
    return BSR.from_blocks(n, b, np.concatenate(rows), np.concatenate(cols), np.concatenate(vals))


def test_upload_staging_is_given_back_when_memory_runs_out():
    H = ring_blocks(6000, 13, 6, 1)  # 105 MB of values
    x = np.random.default_rng(2).standard_normal((H.n_rows, 2))
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        y = ctx.bsr_mult(_lib.SLOT_H, x)
        held = ctx.mem_info()[0]
        with pytest.raises(_lib.RsatbGpuError):
            ctx.set_samples(1 << 31, 256, _lib.SAMPLES_RADEMACHER, 1)  # 4 TB: no card has it
        # the staging of the values, counted in whole granules of at most 2 MB
        assert ctx.mem_info()[0] - held >= H.values.nbytes - 2 * MB
        # and the context goes on
        assert np.array_equal(ctx.bsr_mult(_lib.SLOT_H, x), y)
        ctx.upload_bsr(_lib.SLOT_S, H)
        assert np.array_equal(ctx.bsr_mult(_lib.SLOT_S, x), y)


def test_projected_run_without_room_for_its_stores(monkeypatch):
    """With no room for the chunk dots and dot partials of all steps a projected
    run finishes step by step: the same sums in the same order."""
    H = ring_blocks(4096, 9, 3, 3)
    a = 1.1 * 9 * 7 * 3.0  # above the row sums' scale: any window does
    groups = np.arange(H.n_rows) // 9
    out, held = {}, {}
    for limit in (None, str(MB)):
        if limit:
            monkeypatch.setenv("RG_STORE_MAX", limit)
        with _lib.Context(0) as ctx:
            ctx.upload_bsr(_lib.SLOT_H, H)
            ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.0, a)
            ctx.set_samples(H.n_rows, 16, _lib.SAMPLES_RADEMACHER, 5)
            free = ctx.mem_info()[0]
            out[limit] = ctx.kpm_pdos_moments(512, groups, 4096)
            held[limit] = free - ctx.mem_info()[0]
            plain = ctx.kpm_moments(512)
        assert np.array_equal(plain, out[limit][0])
    for x, y in zip(out[None], out[str(MB)]):
        assert np.array_equal(x, y)
    # 4,096 chunks of 48 bytes in each of 257 steps
    assert held[None] - held[str(MB)] > 40 * MB


@pytest.mark.parametrize("G,M,nx", [(2100, 3, 20000), (9, 3, (1 << 20) + 7), (1, 2, (1 << 20) + 1)])
def test_density_takes_bounded_memory(G, M, nx):
    """Many sets, or a grid above a million points, go through the device in
    pieces (128 MB, and what an allocation rounds up to)."""
    rng = np.random.default_rng(G)
    mu = rng.standard_normal((G, M)) + 1j * rng.standard_normal((G, M))
    x = np.linspace(-1.01, 1.01, nx)
    with _lib.Context(0) as ctx:
        free = ctx.mem_info()[0]
        rho = ctx.kpm_density(mu, x, 0.5 / nx)
        assert free - ctx.mem_info()[0] < 160 * MB
    ref = np.stack([_lib.kpm_density(m, x, 0.5 / nx) for m in mu])
    assert np.array_equal(rho, ref)


def test_density_without_room(monkeypatch):
    monkeypatch.setenv("RG_STORE_MAX", "1000")
    rng = np.random.default_rng(4)
    mu = rng.standard_normal((33, 64)) + 1j * rng.standard_normal((33, 64))
    x = np.linspace(-1.01, 1.01, 1000)
    with _lib.Context(0) as ctx:
        free = ctx.mem_info()[0]
        rho = ctx.kpm_density(mu, x, 0.5 / 1000)
        assert ctx.mem_info()[0] == free
    assert np.array_equal(rho, np.stack([_lib.kpm_density(m, x, 0.5 / 1000) for m in mu]))
