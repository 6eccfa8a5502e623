"""Workloads of this framework's main path, for timing and for checks against 64-bit results.

The tasks are the ones a program calls: the density of states of p_z sheets (one orbital per atom) and of
LCAO-like diamond (9 or 13 orbitals per atom), orthogonal and with an overlap, at Gamma and at k-points, in both
precisions; the projected density; a new structure from its host matrices to moments; the gradient of the
moments; the conductivity spectrum. Sizes are this repository's own configurations or lie around them. Every
structure is periodic and carries disorder drawn from the seed.

listed() and draw() give cases (dicts of plain values), prepare() what a program holds before the call, run() one
pass through the public entry points, exact() the same results from plain torch and numpy in 64 bits, work() the
bytes and operations that a pass cannot do without.
"""
from __future__ import annotations

import functools
import math

import numpy as np
import torch
import torch.utils.checkpoint

from rsatb_amd import _lib
from rsatb_amd.autograd import DifferentiableKPM, LinearOperatorModel
from rsatb_amd.bsr import BSR
from rsatb_amd.driver import PreconditionerOptions, RSATB, SetupOptions
from rsatb_amd.lattice import Edges, Structure

PZ_WINDOW = (-12.5, 12.5)      # holds every p_z spectrum below
PZ_S_WINDOW = (-20.0, 20.0)    # with the nearest-neighbour overlap
LCAO_WINDOW = (-14.0, 14.0)    # 9 or 13 random orbitals, with or without overlap
SHELLS = {1: ((1.5, -2.7),), 3: ((1.5, -2.7), (2.5, -0.25), (2.9, -0.18))}  # (radius, hopping): 3 and 12 bonds an atom


def listed():
    return [
        # a small p_z cell, as in a unit-cell scan: launches and the host's share decide
        {"name": "dos_pz_cell", "kind": "dos_pz", "nx": 12, "ny": 7, "shells": 1, "R": 16, "M": 512, "fp32": False},
        # the plain-DOS configuration: graphene 64 x 64, R = 16, 1024 moments, density included
        {"name": "dos_pz_64", "kind": "dos_pz", "nx": 64, "ny": 64, "shells": 1, "R": 16, "M": 1024, "fp32": False},
        # its scale-up past every cache
        {"name": "dos_pz_sheet", "kind": "dos_pz", "nx": 512, "ny": 512, "shells": 1, "R": 16, "M": 256, "fp32": False},
        # a third-neighbour sheet of odd sides with ten random-phase vectors
        {"name": "dos_pz_phase10", "kind": "dos_pz", "nx": 131, "ny": 113, "shells": 3, "R": 10, "M": 256, "fp32": False,
         "phase": True},
        # the precision form on a large sheet of odd sides
        {"name": "dos_pz_fp32", "kind": "dos_pz", "nx": 401, "ny": 299, "shells": 3, "R": 32, "M": 256, "fp32": True},
        # the non-orthogonal diamond configuration: 8^3 cells, 13 orbitals, R = 64 complex
        {"name": "dos_lcao_64", "kind": "dos_lcao", "nx": 8, "ny": 8, "nz": 8, "b": 13, "vac": 0.0, "R": 64, "M": 128,
         "fp32": False},
        # its precision form at the width of the largest configuration
        {"name": "dos_lcao_fp32", "kind": "dos_lcao", "nx": 10, "ny": 10, "nz": 10, "b": 13, "vac": 0.0, "R": 128,
         "M": 64, "fp32": True},
        # a defective crystal (ragged rows) with few samples, from host matrices to moments: upload, overlap factor,
        # spectral bounds, moments; what every new structure of a series costs
        {"name": "setup_lcao", "kind": "setup", "nx": 7, "ny": 6, "nz": 5, "b": 13, "vac": 0.05, "R": 20, "M": 64,
         "steps": 60},
        # two k-points of a 9-orbital crystal through the driver (complex operators)
        {"name": "dos_kpoints", "kind": "dos_k", "nx": 6, "ny": 5, "nz": 5, "b": 9, "R": 16, "M": 128},
        # projected density on every atom through the driver
        {"name": "pdos_atoms", "kind": "pdos", "nx": 5, "ny": 4, "nz": 4, "b": 9, "R": 16, "M": 256},
        # moments and their gradient with a learnable overlap: graphene 128 x 128, R = 32, checkpoints every 32
        {"name": "grad_pz", "kind": "grad", "nx": 128, "ny": 128, "R": 32, "M": 128, "stride": 32},
        # the conductivity spectrum of a graphene sheet: R = 16, Greenwood
        {"name": "dc_pz", "kind": "dc", "nx": 128, "ny": 128, "shells": 1, "R": 16, "M": 256, "fp32": False},
    ]


def draw(rng):
    def log_int(lo, hi):
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    kind = rng.choice(["dos_pz", "dos_pz", "dos_pz", "dos_lcao", "dos_lcao", "setup", "dos_k", "pdos", "grad", "dc"])
    if kind == "dos_pz":
        fp32 = rng.random() < 0.3
        shells = rng.choice([1, 3])
        R = rng.choice([16, 32]) if fp32 else rng.choice([1, 4, 7, 10, 16, 24, 32])
        phase = rng.random() < 0.4
        side = min(512, int(math.sqrt(2.0e7 / (R * (4 if shells == 3 else 1) * (2 if phase else 1)))))
        nx, ny = log_int(6, side), log_int(6, side)
        return {"kind": kind, "nx": nx, "ny": ny, "shells": shells, "R": R, "M": rng.randint(130, 257), "fp32": fp32,
                "phase": phase}
    if kind == "dos_lcao":
        fp32 = rng.random() < 0.4
        R = rng.choice([32, 64, 128]) if fp32 else rng.choice([8, 10, 16, 24, 32, 50, 64])
        return {"kind": kind, "nx": rng.randint(3, 8), "ny": rng.randint(3, 8), "nz": rng.randint(3, 8),
                "b": rng.choice([9, 13]), "vac": rng.choice([0.0, 0.04]), "R": R, "M": rng.randint(24, 64),
                "fp32": fp32}
    if kind == "setup":
        return {"kind": kind, "nx": rng.randint(3, 7), "ny": rng.randint(3, 6), "nz": rng.randint(3, 5),
                "b": rng.choice([9, 13]), "vac": rng.choice([0.0, 0.05]), "R": rng.choice([8, 16, 20, 32]),
                "M": rng.randint(24, 64), "steps": rng.randint(30, 60)}
    if kind == "dos_k":
        return {"kind": kind, "nx": rng.randint(2, 6), "ny": rng.randint(2, 5), "nz": rng.randint(2, 5),
                "b": rng.choice([9, 13]), "R": rng.choice([4, 8, 16]), "M": rng.randint(60, 128)}
    if kind == "pdos":
        return {"kind": kind, "nx": rng.randint(2, 5), "ny": rng.randint(2, 4), "nz": rng.randint(2, 4),
                "b": rng.choice([9, 13]), "R": rng.choice([4, 10, 16]), "M": rng.randint(100, 256)}
    if kind == "grad":
        return {"kind": kind, "nx": log_int(16, 128), "ny": log_int(16, 128), "R": rng.choice([8, 10, 16, 32]),
                "M": rng.randint(48, 128), "stride": rng.choice([8, 16, 32])}
    return {"kind": kind, "nx": log_int(16, 128), "ny": log_int(16, 128), "shells": rng.choice([1, 3]),
            "R": rng.choice([4, 8, 10, 16]), "M": rng.randint(64, 256), "fp32": False}


# ------------------------------------------------------------------ structures
GRAPHENE = (np.array([[0, 0, 0], [0, 1.42, 0], [0.5 * 3 ** 0.5 * 1.42, 2.13, 0], [0.5 * 3 ** 0.5 * 1.42, 3.55, 0]]),
            np.diag([3 ** 0.5 * 1.42, 4.26, 20.0]))
_FCC = np.array([[0, 0, 0], [0, 0.5, 0.5], [0.5, 0, 0.5], [0.5, 0.5, 0]])
DIAMOND = (np.concatenate([_FCC, _FCC + 0.25]) * 3.567, np.eye(3) * 3.567)


@functools.lru_cache(maxsize=4)
def bonds(lattice, cutoff, nx, ny, nz):
    """Half of the bonds of a periodic supercell, each pair once: (positions, cell, src, dst, shift, vec)."""
    unit, ucell = {"graphene": GRAPHENE, "diamond": DIAMOND}[lattice]
    reps, ns = (nx, ny, nz), len(unit)
    span = [range(-3, 4)] * 2 + [range(-2, 3) if lattice == "diamond" else range(1)]
    cells = np.stack(np.meshgrid(*[np.arange(n) for n in reps], indexing="ij"), -1).reshape(-1, 3)
    pos = (cells[:, None, :] @ ucell + unit[None]).reshape(-1, 3)
    out = [[], [], [], []]
    for a in range(ns):
        for c in range(ns):
            for d in np.stack(np.meshgrid(*span, indexing="ij"), -1).reshape(-1, 3):
                v = unit[c] + d @ ucell - unit[a]
                if not 1e-6 < np.linalg.norm(v) <= cutoff or tuple(v.round(6)) < (0.0, 0.0, 0.0):
                    continue
                to = cells + d
                sh = to // np.array(reps)
                to = to - sh * np.array(reps)
                out[0].append(np.arange(len(cells)) * ns + a)
                out[1].append(((to[:, 0] * ny + to[:, 1]) * nz + to[:, 2]) * ns + c)
                out[2].append(sh)
                out[3].append(np.broadcast_to(v, (len(cells), 3)))
    return (pos, ucell * np.array(reps, dtype=float)[:, None]) + tuple(np.concatenate(x) for x in out)


def both_ways(src, dst, blocks):
    """(rows, cols, blocks) of the symmetric matrix whose half is given."""
    return (np.concatenate([src, dst]), np.concatenate([dst, src]),
            np.concatenate([blocks, np.conj(np.swapaxes(blocks, 1, 2))]))


def with_diagonal(n, diag, half):
    rows, cols, blocks = half
    i = np.arange(n)
    return np.concatenate([i, rows]), np.concatenate([i, cols]), np.concatenate([diag.astype(blocks.dtype), blocks])


@functools.lru_cache(maxsize=2)
def pz_sheet(nx, ny, shells, seed):
    """H of a graphene sheet with onsite disorder and bond modulation, and its three bond moments B_a."""
    rng = np.random.default_rng(seed)
    _, _, src, dst, _, vec = bonds("graphene", SHELLS[shells][-1][0], nx, ny, 1)
    n = 4 * nx * ny
    r = np.linalg.norm(vec, axis=1)
    t = np.zeros(src.size)
    for radius, hop in reversed(SHELLS[shells]):
        t[r <= radius] = hop
    u = rng.uniform(-1, 1, n)
    t = (t * (1.0 + 0.03 * (u[src] + u[dst])))[:, None, None]
    H = with_diagonal(n, rng.uniform(-0.8, 0.8, n)[:, None, None], both_ways(src, dst, t))
    zero = np.zeros((n, 1, 1))
    B = []
    for a in range(3):
        w = t * vec[:, a, None, None]
        rows, cols, _ = both_ways(src, dst, t)
        B.append(with_diagonal(n, zero, (rows, cols, np.concatenate([w, -w]))))
    return n, H, B


@functools.lru_cache(maxsize=2)
def lcao(nx, ny, nz, b, vac, seed):
    """Half the bonds with random blocks of H and S, and the onsite blocks, of diamond with vacancies."""
    rng = np.random.default_rng(seed)
    pos, cell, src, dst, shift, vec = bonds("diamond", 2.7, nx, ny, nz)
    keep = rng.random(len(pos)) >= vac
    number = np.cumsum(keep) - 1
    on = keep[src] & keep[dst]
    src, dst, shift, vec = number[src[on]], number[dst[on]], shift[on], vec[on]
    n = int(keep.sum())
    decay = np.exp(-np.linalg.norm(vec, axis=1) / 1.5)[:, None, None]
    h = rng.standard_normal((src.size, b, b)) * decay
    s = rng.standard_normal((src.size, b, b)) * (0.05 * decay)
    d = rng.standard_normal((n, b, b))
    return {"n": n, "pos": pos[keep], "cell": cell, "src": src, "dst": dst, "shift": shift, "vec": vec, "h": h,
            "s": s, "h0": np.triu(d) + np.swapaxes(np.triu(d, 1), 1, 2)}


def lcao_matrix(m, which, k=None):
    blocks = m["h" if which == "H" else "s"]
    if k is not None:
        blocks = blocks * np.exp(2j * np.pi * (m["shift"] @ np.asarray(k)))[:, None, None]
    diag = m["h0"] if which == "H" else np.broadcast_to(np.eye(blocks.shape[1]), m["h0"].shape)
    return with_diagonal(m["n"], diag, both_ways(m["src"], m["dst"], blocks))


def to_bsr(n, entries):
    rows, cols, blocks = entries
    return BSR.from_blocks(n, blocks.shape[1], rows, cols, blocks)


def sample_block(rows, R, phase, seed):
    rng = np.random.default_rng(seed + 77)
    if phase:
        return np.exp(2j * np.pi * rng.random((rows, R))) / math.sqrt(rows)
    return (2.0 * rng.integers(0, 2, (rows, R)) - 1.0) / math.sqrt(rows)


class Crystal:
    """The model of an orthogonal LCAO crystal as the driver takes one."""

    cutoff = 2.7

    def __init__(self, m):
        self.m, self.norb = m, m["h"].shape[1]
        self.structure = Structure(m["pos"], m["cell"])
        src, dst, _ = both_ways(m["src"], m["dst"], m["h"])
        vec = np.concatenate([m["vec"], -m["vec"]])
        self.edges = Edges(src, dst, np.concatenate([m["shift"], -m["shift"]]), vec, np.linalg.norm(vec, axis=1))

    def has_overlap(self):
        return False

    def blocks(self, st, edges, which):
        return self.m["h0"], both_ways(self.m["src"], self.m["dst"], self.m["h"])[2]


def resolution(window, M):
    """The dE for which the DOS task takes M moments."""
    return math.sqrt(8.0 * math.log(2.0)) * math.pi * 0.5 * (window[1] - window[0]) / (M - 0.5)


# ------------------------------------------------------------------ the gradient's model
def grad_model(c):
    """theta = (e0, t1, t2, t3, s1) of a sheet: every coefficient's matrix on one pattern, for H and for S."""
    _, _, src, dst, _, vec = bonds("graphene", 2.9, c["nx"], c["ny"], 1)
    n, r = 4 * c["nx"] * c["ny"], np.linalg.norm(vec, axis=1)
    one, zero = np.ones((n, 1, 1)), np.zeros((n, 1, 1))
    H = [with_diagonal(n, one, both_ways(src, dst, np.zeros((src.size, 1, 1))))]
    lo = 0.0
    for radius, _ in SHELLS[3]:
        H.append(with_diagonal(n, zero, both_ways(src, dst, ((r > lo) & (r <= radius)).astype(float)[:, None, None])))
        lo = radius
    near = r <= 1.5
    src, dst = src[near], dst[near]
    S = [with_diagonal(n, one, both_ways(src, dst, np.zeros((src.size, 1, 1)))),
         with_diagonal(n, zero, both_ways(src, dst, np.ones((src.size, 1, 1))))]
    return n, H, S


def grad_inputs(c, seed):
    rng = np.random.default_rng(seed)
    theta = np.array([0.2, -2.7, -0.25, -0.18, 0.1]) * (1.0 + 0.05 * rng.uniform(-1, 1, 5))
    return theta, rng.standard_normal(c["M"]) / np.sqrt(1.0 + np.arange(c["M"]))


# ------------------------------------------------------------------ prepare and run
def prepare(case, seed):
    c = dict(case)
    kind = c["kind"]
    st = {"c": c}
    if kind in ("dos_k", "pdos"):
        model = Crystal(lcao(c["nx"], c["ny"], c["nz"], c["b"], 0.0, seed))
        points = [[0.0, 0.0, 0.0]] if kind == "pdos" else [[0.13, -0.21, 0.07], [0.3, 0.1, -0.4]]
        st["calc"] = RSATB(model.structure, model, SetupOptions(kpoints=points, nsamples=c["R"], sample_seed=seed,
                                                                energy_bounds=LCAO_WINDOW), edges=model.edges)
        st["calc"].context.set_samples(model.m["n"] * c["b"], c["R"], _lib.SAMPLES_UPLOAD_COMPLEX,
                                       data=sample_block(model.m["n"] * c["b"], c["R"], True, seed))
        return st
    if kind == "grad":
        n, H, S = grad_model(c)
        H, S = [to_bsr(n, x) for x in H], [to_bsr(n, x) for x in S]
        basis = np.stack([x.values.reshape(-1) for x in H], 1)
        st["engine"] = DifferentiableKPM(
            LinearOperatorModel(H[0], basis, ("e0", "t1", "t2", "t3")), c["R"], PZ_S_WINDOW, c["M"], c["stride"],
            overlap=LinearOperatorModel(S[0], S[1].values.reshape(-1, 1), ("s1",), offset=S[0].values.reshape(-1)))
        st["engine"].ctx.set_samples(n, c["R"], _lib.SAMPLES_UPLOAD_COMPLEX, data=sample_block(n, c["R"], True, seed))
        st["theta"], st["g"] = grad_inputs(c, seed)
        return st
    ctx = st["ctx"] = _lib.Context()
    if kind == "dos_pz" or kind == "dc":
        n, H, B = pz_sheet(c["nx"], c["ny"], c["shells"], seed)
        rows, phase, form, window = n, c.get("phase", False), _lib.FORM_ORTHOGONAL, PZ_WINDOW
        ctx.upload_bsr(_lib.SLOT_H, to_bsr(n, H))
        for a in range(3 if kind == "dc" else 0):
            ctx.upload_bsr(_lib.SLOT_VX + a, to_bsr(n, B[a]))
    else:
        m = lcao(c["nx"], c["ny"], c["nz"], c["b"], c["vac"], seed)
        rows, phase, form, window = m["n"] * c["b"], True, _lib.FORM_SANDWICH, LCAO_WINDOW
        H, S = to_bsr(m["n"], lcao_matrix(m, "H")), to_bsr(m["n"], lcao_matrix(m, "S"))
        if kind == "setup":
            st["H"], st["S"] = H, S
        else:
            ctx.upload_bsr(_lib.SLOT_S, S)
            ctx.isqrt_patches()
            ctx.upload_bsr(_lib.SLOT_H, H)
    st["window"] = window
    ctx.set_operator(form, 0.5 * (window[0] + window[1]), 0.5 * (window[1] - window[0]))
    ctx.set_samples(rows, c["R"], _lib.SAMPLES_UPLOAD_COMPLEX if phase else _lib.SAMPLES_UPLOAD_REAL,
                    data=sample_block(rows, c["R"], phase, seed))
    return st


def run(st):
    c = st["c"]
    kind = c["kind"]
    prec = _lib.PREC_FP32 if c.get("fp32") else _lib.PREC_FP64
    if kind == "dos_pz":
        dos, energy = st["ctx"].compute_dos(*st["window"], resolution(st["window"], c["M"]), prec)
        return {"dos": dos, "energy": energy}
    if kind == "dos_lcao":
        mu, cols = st["ctx"].kpm_moments(c["M"], prec, per_column=True)
        return {"mu": mu, "columns": cols}
    if kind == "setup":
        ctx = st["ctx"]
        ctx.upload_bsr(_lib.SLOT_S, st["S"])
        ctx.isqrt_patches()
        ctx.upload_bsr(_lib.SLOT_H, st["H"])
        bounds = ctx.estimate_bounds(_lib.FORM_SANDWICH, steps=c["steps"])
        mu, cols = ctx.kpm_moments(c["M"], per_column=True)
        return {"bounds": np.array(bounds), "mu": mu, "columns": cols}
    if kind == "dos_k":
        dos, energy = st["calc"].compute_dos(resolution(LCAO_WINDOW, c["M"]))
        return {"dos": dos, "energy": energy}
    if kind == "pdos":
        out = st["calc"].compute_pdos(resolution(LCAO_WINDOW, c["M"]), "atom")
        return {"energy": out["energy"], "pdos": out["pdos"], "total": out["total"]}
    if kind == "grad":
        mu = st["engine"].forward(st["theta"])
        return {"mu": mu, "grad": st["engine"].backward(st["g"])}
    sigma, energy, mu = st["ctx"].dc_spectrum(c["M"], with_moments=True, precision=prec)
    return {"sigma": sigma, "energy": energy, "mu": mu}


# ------------------------------------------------------------------ the same in plain 64-bit torch
def _dev():
    return "cuda" if torch.cuda.is_available() else "cpu"


def product(n, entries):
    """x -> A x for [rows, W] tensors."""
    rows, cols, blocks = entries
    b = blocks.shape[1]
    if b == 1:
        A = torch.sparse_coo_tensor(torch.from_numpy(np.stack([rows, cols])), torch.from_numpy(blocks.reshape(-1)),
                                    (n, n)).coalesce().to_sparse_csr().to(_dev())
        return lambda x: torch.view_as_complex((A @ torch.view_as_real(x).reshape(n, -1)).reshape(n, -1, 2)) \
            if x.is_complex() else A @ x
    r, q, v = (torch.from_numpy(np.ascontiguousarray(t)).to(_dev()) for t in (rows, cols, blocks))

    def apply(x):
        xr = x
        if x.is_complex() and not v.is_complex():
            xr = torch.view_as_real(x).reshape(x.shape[0], -1)
        xr = xr.reshape(n, b, -1)
        y = torch.zeros_like(xr)
        for k in range(0, len(r), 65536):
            y.index_add_(0, r[k:k + 65536], torch.bmm(v[k:k + 65536], xr[q[k:k + 65536]].contiguous()))
        y = y.reshape(n * b, -1)
        return torch.view_as_complex(y.reshape(n * b, -1, 2)) if x.is_complex() and not v.is_complex() else y

    return apply


def overlap_factor(n, entries, steps=18):
    """Entries of Z: block row i is block i's rows of S[C_i, C_i]^(-1/2), C_i the stored columns of row i."""
    rows, cols, blocks = entries
    b = blocks.shape[1]
    key, at = np.unique(rows.astype(np.int64) * n + cols, return_inverse=True)
    v = torch.zeros(len(key) + 1, b, b, dtype=torch.float64, device=_dev())
    v.index_add_(0, torch.from_numpy(at).to(_dev()), torch.from_numpy(np.ascontiguousarray(blocks)).to(_dev()))
    urow, ucol = key // n, key % n
    ptr = np.searchsorted(urow, np.arange(n + 1))
    most = int(np.max(np.diff(ptr)))
    place = np.arange(len(key)) - ptr[urow]
    nb = np.full((n, most), -1)
    nb[urow, place] = ucol
    out = torch.zeros_like(v[:-1])
    for lo in range(0, n, 1024):
        p = nb[lo:lo + 1024]
        pair = np.where((p[:, :, None] >= 0) & (p[:, None, :] >= 0), p[:, :, None] * n + p[:, None, :], -1)
        idx = np.minimum(np.searchsorted(key, pair), len(key) - 1)
        idx = np.where(key[idx] == pair, idx, len(key))
        A = v[torch.from_numpy(idx).to(v.device)].permute(0, 1, 3, 2, 4).reshape(len(p), most * b, most * b)
        pad = torch.from_numpy(np.repeat(p < 0, b, 1)).to(v.device)
        A = A + torch.diag_embed(pad.double())
        scale = A.abs().sum(2).amax(1)[:, None, None]
        eye = torch.eye(most * b, dtype=torch.float64, device=v.device)
        Y, Z = A / scale, eye.expand_as(A).contiguous()
        for _ in range(steps):
            T = 1.5 * eye - 0.5 * torch.bmm(Z, Y)
            Y, Z = torch.bmm(Y, T), torch.bmm(T, Z)
        Z = (Z / scale.sqrt()).reshape(len(p), most, b, most, b)
        s = np.arange(ptr[lo], ptr[lo + len(p)])
        i = urow[s] - lo
        own = np.argmax(p == (np.arange(len(p)) + lo)[:, None], 1)
        out[torch.from_numpy(s).to(v.device)] = Z[torch.from_numpy(i), torch.from_numpy(own[i]), :,
                                                  torch.from_numpy(place[s]), :]
    return urow, ucol, out.cpu().numpy()


def window_op(apply, window):
    a, c = 0.5 * (window[1] - window[0]), 0.5 * (window[0] + window[1])
    return lambda x: (apply(x) - c * x) / a


def moments(op, psi, M, dot):
    """[M, ...] moments from the doubled recurrence; dot(x, y) the inner products <x|y> that are wanted."""
    t0, t1 = psi, op(psi)
    m0, m1 = dot(t0, t0), dot(t0, t1)
    mu = [m0, m1, 2 * dot(t1, t1) - m0]
    while len(mu) < M:
        t0, t1 = t1, 2 * op(t1) - t0
        mu += [2 * dot(t1, t0) - m1, 2 * dot(t1, t1) - m0]
    return torch.stack(mu[:M])


def columns(x, y):
    return (x.conj() * y).sum(0).to(torch.complex128)


def jackson(M):
    i, d = np.arange(M), M + 1.0
    return ((d - i) * np.cos(np.pi * i / d) + np.sin(np.pi * i / d) / np.tan(np.pi / d)) / d


def density(mu, window, M):
    """2 rho of [..., M] moments on the DOS task's grid, and its energies."""
    half, mid = 0.5 * (window[1] - window[0]), 0.5 * (window[0] + window[1])
    nt = max(1, math.ceil((window[1] - window[0]) / resolution(window, M)))
    g = np.concatenate([(np.arange(nt) - nt) / nt, np.arange(nt) / nt])
    x = np.clip(g, -1 + 0.5 / nt, 1 - 0.5 / nt)
    w = jackson(M) * np.where(np.arange(M) == 0, 1.0, 2.0)
    T = np.cos(np.arange(M)[:, None] * np.arccos(x)[None])
    return 2.0 * ((mu.real * w) @ T) / (np.pi * np.sqrt(np.maximum(1e-14, 1 - x * x))), g * half + mid


def psi_of(rows, R, phase, seed):
    return torch.from_numpy(sample_block(rows, R, phase, seed)).to(_dev())


def exact(case, seed):
    c = dict(case)
    kind, M, R = c["kind"], c["M"], c["R"]
    if kind == "dos_pz":
        n, H, _ = pz_sheet(c["nx"], c["ny"], c["shells"], seed)
        mu = moments(window_op(product(n, H), PZ_WINDOW), psi_of(n, R, c.get("phase", False), seed), M, columns)
        dos, energy = density(mu.mean(1).cpu().numpy(), PZ_WINDOW, M)
        return {"dos": dos, "energy": energy}
    if kind in ("dos_lcao", "setup"):
        m = lcao(c["nx"], c["ny"], c["nz"], c["b"], c["vac"], seed)
        ur, uc, z = overlap_factor(m["n"], lcao_matrix(m, "S"))
        Z, H = product(m["n"], (ur, uc, z)), product(m["n"], lcao_matrix(m, "H"))
        Zt = product(m["n"], (uc, ur, np.ascontiguousarray(np.swapaxes(z, 1, 2))))
        cols = moments(window_op(lambda x: Zt(H(Z(x))), LCAO_WINDOW), psi_of(m["n"] * c["b"], R, True, seed), M,
                       columns)
        out = {"mu": cols.mean(1), "columns": cols}
        # the bounds are Ritz values after a fixed number of steps: no value of their own
        return {"bounds": None, **out} if kind == "setup" else out
    if kind == "dos_k":
        m, parts = lcao(c["nx"], c["ny"], c["nz"], c["b"], 0.0, seed), []
        for k in ([0.13, -0.21, 0.07], [0.3, 0.1, -0.4]):
            op = window_op(product(m["n"], lcao_matrix(m, "H", k)), LCAO_WINDOW)
            mu = moments(op, psi_of(m["n"] * c["b"], R, True, seed), M, columns).mean(1)
            dos, energy = density(mu.cpu().numpy(), LCAO_WINDOW, M)
            parts.append(dos)
        return {"dos": np.concatenate(parts), "energy": energy}
    if kind == "pdos":
        m = lcao(c["nx"], c["ny"], c["nz"], c["b"], 0.0, seed)
        n, b = m["n"], c["b"]
        mu = moments(window_op(product(n, lcao_matrix(m, "H")), LCAO_WINDOW), psi_of(n * b, R, True, seed), M,
                     lambda x, y: (x.conj() * y).reshape(n, -1).sum(1))
        mu = (mu / R).cpu().numpy().T
        pdos, energy = density(mu, LCAO_WINDOW, M)
        return {"energy": energy, "pdos": pdos[None], "total": density(mu.sum(0), LCAO_WINDOW, M)[0][None]}
    if kind == "grad":
        return exact_grad(c, seed)
    n, H, B = pz_sheet(c["nx"], c["ny"], c["shells"], seed)
    op = window_op(product(n, H), PZ_WINDOW)
    psi, a = psi_of(n, R, False, seed), 0.5 * (PZ_WINDOW[1] - PZ_WINDOW[0])

    def chain(x):
        t0, t1 = x, op(x)
        yield t0
        for _ in range(M - 1):
            yield t1
            t0, t1 = t1, 2 * op(t1) - t0

    mu = torch.zeros(3, M, M, dtype=torch.float64, device=psi.device)
    for d in range(3):
        V = product(n, B[d])
        left = torch.stack([V(t).reshape(-1) for t in chain(psi)])
        right = torch.stack([t.reshape(-1) for t in chain(V(psi))])
        mu[d] = left @ right.T / (4 * a * a)
    mu = mu.cpu().numpy()
    th = np.pi * (np.arange(M) + 0.5) / M
    W = (2 * jackson(M) / np.pi / np.where(np.arange(M) == 0, 2.0, 1.0))[:, None] * np.cos(np.outer(np.arange(M), th))
    sigma = np.zeros((M, 6))
    for d, at in enumerate((0, 3, 5)):
        sigma[:, at] = ((W * (mu[d] @ W)).sum(0) / np.maximum(1e-14, np.sin(th) ** 2) / R)[::-1]
    return {"sigma": sigma, "energy": (a * np.cos(th))[::-1] + 0.5 * sum(PZ_WINDOW), "mu": mu.astype(complex)}


def exact_grad(c, seed):
    """Moments and dL/dtheta by torch's own autograd through S -> Z and the recurrence."""
    n, H, S = grad_model(c)
    theta, g = grad_inputs(c, seed)
    th = torch.tensor(theta, device=_dev(), requires_grad=True)

    def pattern(mats):
        """Neighbour table [n, k] of a uniform pattern and each matrix's values on it."""
        rows, cols = mats[0][0], mats[0][1]
        key, at = np.unique(rows.astype(np.int64) * n + cols, return_inverse=True)
        k = np.bincount(key // n, minlength=n)
        if k.min() != k.max():
            return None
        vals = [np.bincount(at, m[2].reshape(-1), len(key)).reshape(n, -1) for m in mats]
        return (torch.from_numpy((key % n).reshape(n, -1)).to(_dev()),
                [torch.from_numpy(v).to(_dev()) for v in vals])

    hp, sp = pattern(H), pattern(S)
    if hp is None or sp is None:
        return None
    hn, hv = hp
    sn, sv = sp
    h = sum(v * th[i] for i, v in enumerate(hv))
    s = sv[0] + th[4] * sv[1]
    k = sn.shape[1]
    # patch A[i, p, q] = S[C_ip, C_iq]: the stored entry of row C_ip whose column is C_iq, if there is one
    hit = sn[sn][:, :, None, :] == sn[:, None, :, None]
    A = torch.where(hit, s[sn][:, :, None, :], torch.zeros((), dtype=s.dtype, device=s.device)).sum(-1)
    scale = A.detach().abs().sum(2).amax(1)[:, None, None]
    eye = torch.eye(k, dtype=torch.float64, device=s.device)
    Y, Z = A / scale, eye.expand_as(A)
    for _ in range(14):
        T = 1.5 * eye - 0.5 * (Z[:, :, :, None] * Y[:, None, :, :]).sum(2)
        Y, Z = (Y[:, :, :, None] * T[:, None, :, :]).sum(2), (T[:, :, :, None] * Z[:, None, :, :]).sum(2)
    own = (sn == torch.arange(n, device=s.device)[:, None]).double()
    z = (own[:, :, None] * (Z / scale.sqrt())).sum(1)
    back = (sn[sn] == torch.arange(n, device=s.device)[:, None, None])  # [n, k, k]: where row C_ip stores column i
    zt = torch.where(back, z[sn], torch.zeros((), dtype=s.dtype, device=s.device)).sum(-1)

    def apply(vals, nb, x):
        y = vals[:, 0, None] * x[nb[:, 0]]
        for j in range(1, nb.shape[1]):
            y = y + vals[:, j, None] * x[nb[:, j]]
        return y

    op = window_op(lambda x: apply(zt, sn, apply(h, hn, apply(z, sn, x))), PZ_S_WINDOW)
    step = lambda x, y: torch.utils.checkpoint.checkpoint(lambda u, v: 2 * op(u) - v, x, y, use_reentrant=False)  # noqa: E731
    psi = psi_of(n, c["R"], True, seed)
    dot = lambda x, y: (x.conj() * y).sum().real / c["R"]  # noqa: E731
    t0, t1 = psi, op(psi)
    m0, m1 = dot(t0, t0), dot(t0, t1)
    mu = [m0, m1, 2 * dot(t1, t1) - m0]
    while len(mu) < c["M"]:
        t0, t1 = t1, step(t1, t0)
        mu += [2 * dot(t1, t0) - m1, 2 * dot(t1, t1) - m0]
    mu = torch.stack(mu[:c["M"]])
    (mu * torch.tensor(g, device=mu.device)).sum().backward()
    return {"mu": mu.detach(), "grad": th.grad}


def work(case):
    """Per operator product: its matrix once and each vector that it reads or writes once, as the recurrence needs
    them (three vectors a step; two more for every further factor of a sandwich)."""
    c = dict(case)
    kind, R, M = c["kind"], c["R"], c["M"]
    steps, eb = M // 2, 4 if c.get("fp32") else 8
    if kind in ("dos_pz", "grad", "dc"):
        n, b = 4 * c["nx"] * c["ny"], 1
        per = {1: 4, 3: 13}[c.get("shells", 3)]
    else:
        n, b = 8 * c["nx"] * c["ny"] * c["nz"], c["b"]
        per = 17
        n = int(n * (1 - c.get("vac", 0.0)))
        per = 1 + 16 * (1 - c.get("vac", 0.0))
    cv = 2 if c.get("phase") or kind not in ("dos_pz", "dc") else 1
    cm = 2 if kind == "dos_k" else 1
    mat = n * per * (b * b * eb * cm + 4)
    flop = 2.0 * n * per * b * b * R * cv * cm
    vec = n * b * R * eb * cv
    if kind == "dos_pz":
        return {"bytes": steps * (mat + 3 * vec), "flops": steps * flop}
    if kind == "dos_k":
        return {"bytes": 2 * steps * (mat + 3 * vec), "flops": 2 * steps * flop}
    if kind == "pdos":
        return {"bytes": steps * (mat + 3 * vec) + 8.0 * n * M, "flops": steps * flop + 2.0 * n * M * 0.28 * M}
    if kind == "dos_lcao":
        return {"bytes": steps * (3 * mat + 7 * vec), "flops": 3 * steps * flop}
    if kind == "setup":
        dim = per * b
        chain = 3 * mat + 7 * n * b * 16 * 8
        return {"bytes": steps * (3 * mat + 7 * vec) + c["steps"] * chain + 4 * mat,
                "flops": 3 * (steps + c["steps"] * 16.0 / (2 * R)) * flop + 18 * 2.0 * n * dim ** 3}
    if kind == "grad":
        zmat = n * 4 * 12
        chain = 2 * zmat + mat + 7 * vec
        pattern = n * 17 * 8 + 4 * vec
        return {"bytes": steps * (3 * chain + pattern), "flops": 3 * steps * flop * 21 / 13 + steps * flop * 21 / 13}
    # conductivity: one base and three right recurrences, three velocity products a moment, one contraction an axis
    return {"bytes": M * (4 * (mat + 3 * vec) + 3 * (mat + 2 * vec)) + 6 * M * vec,
            "flops": 7 * M * flop + 3 * 2.0 * M * M * n * R}
