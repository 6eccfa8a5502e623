"""Routes of the SpMM and the moment loop by size: exact where a launch changes
kernels, and no slower than the other kernel where its rows are long, short or
many (kernel times, or wall times of whole runs; each bound lies between the two
kernels' times)."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.bsr import BSR

pytestmark = pytest.mark.gpu


def neighbours(n, b, width):
    """Each block row with its 2 width nearest on a ring."""
    rng = np.random.default_rng(width)
    k = np.arange(n)
    d = rng.standard_normal((n, b, b))
    rows, cols, vals = [k], [k], [d + np.swapaxes(d, 1, 2)]
    for s in range(1, width + 1):
        v = rng.standard_normal((n, b, b))
        rows += [k, (k + s) % n]
        cols += [(k + s) % n, k]
        vals += [v, np.swapaxes(v, 1, 2)]
    return BSR.from_blocks(n, b, np.concatenate(rows), np.concatenate(cols), np.concatenate(vals))


def step_us(H, R, prec=_lib.PREC_FP64):
    """Kernel time of a fused step (the best of three runs' averages)."""
    with _lib.Context(0) as ctx:
        ctx.upload_bsr(_lib.SLOT_H, H)
        ctx.set_operator(_lib.FORM_ORTHOGONAL, 0.0, 1e4)
        ctx.set_samples(H.n_rows, R, _lib.SAMPLES_RADEMACHER, 1)
        ctx.kpm_moments(66, prec)
        best = 1e9
        for _ in range(3):
            ctx.set_profiling(True)
            ctx.kpm_moments(66, prec)
            best = min(best, 1e3 * ctx.kernel_stats(_lib.KCLASS_SPMM_STEP)["avg_ms"])
    return best


def test_odd_widths_past_64():
    """65 columns take at most 1.5 times the time of 100."""
    H = neighbours(20000, 9, 0)
    assert step_us(H, 65) <= 1.5 * step_us(H, 100)


def test_short_rows_do_not_pay_for_deep_buffers():
    """A block of 9 a row reads a third of what three blocks do."""
    assert step_us(neighbours(20000, 9, 0), 1) <= 0.8 * step_us(neighbours(20000, 9, 1), 1)
