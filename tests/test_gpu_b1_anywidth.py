"""The slab SpMM of scalar real operators for every row of whole 16-byte pieces
against the column-per-lane layout: widths of one piece, odd and even counts,
a lone row per workgroup, uniform and ragged rows (with empty ones), row counts
that leave the last workgroup and the last XCD range ragged. Products bit for
bit (the same operations in the same order); the moments differ only in the
order of FP64 sums of at most 1,000 rows (1e-12)."""
import numpy as np
import pytest

from rsatb_amd import _lib
from rsatb_amd.autograd import DifferentiableKPM, sk_pz_parameterization
from rsatb_amd.bsr import BSR
from rsatb_amd.lattice import graphene_rect_supercell, neighbor_edges

pytestmark = pytest.mark.gpu


@pytest.fixture
def layout(monkeypatch):
    def use(slab, xcd="1"):
        monkeypatch.setenv("RG_B1V", slab)
        monkeypatch.setenv("RG_B1V_MIN", "0" if slab == "-1" else "-1")  # 0: slabs at every size
        monkeypatch.setenv("RG_XCD_MAP", xcd)
        monkeypatch.setenv("RG_GRAPH", "1")  # the launched loop also where the on-chip one would run

    yield use
    monkeypatch.setenv("RG_B1V", "-1")
    monkeypatch.setenv("RG_B1V_MIN", "-1")
    monkeypatch.setenv("RG_XCD_MAP", "1")
    monkeypatch.delenv("RG_GRAPH", raising=False)
    _lib.Context(0).close()  # the knobs are process-wide


def operator(kind, nbr):
    rng = np.random.default_rng(nbr)
    D = np.zeros((nbr, nbr))
    if kind == "uniform":  # thirteen entries a row
        for k in range(7):
            v = rng.standard_normal(nbr)
            for i in range(nbr):
                D[i, (i + k) % nbr] = D[(i + k) % nbr, i] = v[i]
    else:
        D = np.where(rng.random((nbr, nbr)) < 4.0 / nbr, rng.standard_normal((nbr, nbr)), 0.0)
        D = 0.5 * (D + D.T)
        D[::7] = 0.0
        D[:, ::7] = 0.0  # empty rows
    r, c = np.nonzero(D)
    return BSR.from_blocks(nbr, 1, r, c, D[r, c].reshape(-1, 1, 1)), 1.01 * np.abs(np.linalg.eigvalsh(D)).max()


# (R, complex, FP32): 16-byte pieces a row in the comment
WIDTHS = [
    (2, False, False),    # 1
    (1, True, False),     # 1
    (10, False, False),   # 5
    (7, True, False),     # 7
    (10, True, False),    # 10
    (24, False, False),   # 12
    (12, False, True),    # 3
    (6, True, True),      # 3
    (64, False, False),   # 32
    (70, True, False),    # 70: three rows a workgroup
    (130, True, False),   # 130: one row
    (256, True, False),   # 256: one row, every lane
    (3, False, False),    # no whole pieces: the column-per-lane layout
]


@pytest.mark.parametrize("kind,nbr", [("uniform", 997), ("ragged", 413)])
@pytest.mark.parametrize("R,cplx,fp32", WIDTHS)
def test_any_width_slab_agrees(layout, kind, nbr, R, cplx, fp32):
    H, half = operator(kind, nbr)
    rng = np.random.default_rng(R)
    X = rng.standard_normal((nbr, R))
    if cplx:
        X = X + 1j * rng.standard_normal((nbr, R))
    prec = _lib.PREC_FP32 if fp32 else _lib.PREC_FP64
    out = []
    for slab, xcd in (("0", "1"), ("-1", "1"), ("-1", "0")):
        layout(slab, xcd)
        with _lib.Context(0) as c:
            c.upload_bsr(_lib.SLOT_H, H)
            c.set_operator(_lib.FORM_ORTHOGONAL, 0.1, half + 0.1)
            c.set_samples(nbr, R, _lib.SAMPLES_PHASE if cplx else _lib.SAMPLES_RADEMACHER, 5)
            m = [c.kpm_moments(24, prec, doubling=d) for d in (_lib.DOUBLING_AUTO, _lib.DOUBLING_OFF)]
            Y = c.bsr_mult(_lib.SLOT_H, X)
        out.append((Y, m))
    for Y, m in out[1:]:
        assert np.array_equal(Y, out[0][0])
        for a, b in zip(m, out[0][1]):
            a, b = np.asarray(a), np.asarray(b)
            assert np.max(np.abs(a - b)) <= 1e-12 * np.max(np.abs(b))


@pytest.mark.parametrize("R", [10, 24])
def test_any_width_slab_adjoint_agrees(layout, R):
    # the step that injects three earlier vectors
    st = graphene_rect_supercell(8, 8)
    model = sk_pz_parameterization(st, neighbor_edges(st, 1.6), [1.6])
    grads = []
    for slab in ("0", "-1"):
        layout(slab)
        eng = DifferentiableKPM(model, R, (-8.2, 8.2), 90, checkpoint_stride=8)
        try:
            eng.forward(np.array([0.0, -2.7]))
            grads.append(eng.ctx.kpm_moments_backward(np.linspace(1.0, -1.0, 90)))
        finally:
            eng.ctx.close()
    assert np.max(np.abs(grads[1] - grads[0])) <= 1e-12 * np.max(np.abs(grads[0]))
