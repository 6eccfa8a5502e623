"""The device density reconstruction against the host evaluation, bit for bit:
set counts around the batch of eight, one and several moments, grids around a
wave, grid points past the clamp."""
import numpy as np
import pytest

from rsatb_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,M,nx", [(1, 1, 25000), (1, 2, 12000), (1, 600, 63), (7, 301, 64), (8, 300, 65),
                                    (9, 257, 129), (33, 64, 1000), (3, 2, 5)])
@pytest.mark.parametrize("kernel", [_lib.KERNEL_NONE, _lib.KERNEL_JACKSON, _lib.KERNEL_COSTAPER])
def test_density_equals_host(G, M, nx, kernel):
    rng = np.random.default_rng(G + M)
    mu = rng.standard_normal((G, M)) + 1j * rng.standard_normal((G, M))
    x = np.linspace(-1.01, 1.01, nx)
    with _lib.Context(0) as ctx:
        rho = ctx.kpm_density(mu, x, 0.5 / nx, kernel)
    ref = np.stack([_lib.kpm_density(m, x, 0.5 / nx, kernel) for m in mu])
    assert np.array_equal(rho, ref)
