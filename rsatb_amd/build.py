"""Builds the gfx950 library librsatb_gpu.so in-tree with hipcc.

`python -m rsatb_amd.build` (or `build()`) compiles every HIP source under
rsatb_amd/csrc into one shared object next to this file. The library exports
only the C ABI declared in include/rsatb_gpu.h.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
LIB = PKG / "librsatb_gpu.so"

SOURCES = ["rg_mfma_f64.hip", "rg_mfma_f32.hip", "rg_mfma_cplx.hip", "rg_kernels.hip", "rg_isqrt.hip", "rg_lanczos.hip", "rg_adjoint.hip", "rg_pdos.hip", "rg_density.hip", "rg_onchip.hip", "rg_kg.hip",
           "rg_sk.hip", "rg_engine.hip"]

# -packed-fp32-ops: hipcc generates no packed (v_pk_*) FP32 arithmetic.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    "--offload-arch=gfx950",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fvisibility=hidden",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found: the gfx950 library cannot be built")
    return path


def build(verbose: bool = False, jobs: int = 4) -> Path:
    """Compiles all sources (always) and links librsatb_gpu.so."""
    objdir = PKG / "_build"
    objdir.mkdir(exist_ok=True)
    cc = hipcc()
    procs = []
    objs = []
    for src in SOURCES:
        obj = objdir / (Path(src).stem + ".o")
        objs.append(obj)
        cmd = [cc, *HIPCC_FLAGS, "-I", str(ROOT / "include"), "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    errors = []
    for src, p in procs:
        out, _ = p.communicate()
        text = out.decode(errors="replace")
        if p.returncode != 0:
            errors.append(f"--- {src} ---\n{text}")
        elif verbose and text.strip():
            print(text)
    if errors:
        raise RuntimeError("hipcc failed:\n" + "\n".join(errors))
    tmp = LIB.with_suffix(".so.tmp")
    link = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp), "-lrocblas"]
    if verbose:
        print(" ".join(link), flush=True)
    r = subprocess.run(link, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout.decode(errors="replace"))
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
