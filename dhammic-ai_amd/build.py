"""Build libssd_mi355x.so for gfx950 from csrc/*.hip with hipcc.

    python dhammic-ai_amd/build.py [--jobs N] [--verbose]

Objects go to dhammic-ai_amd/_build/, the library to
dhammic-ai_amd/kernels/libssd_mi355x.so (in-tree, so it travels with the
source tree to the GPU box).
"""
from __future__ import annotations

import argparse
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "kernels" / "libssd_mi355x.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-mcode-object-version=5",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable", "-Wno-unused-parameter",
    # packed fp32 VALU ops are kept out of every kernel (some of their forms have given wrong results)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{PKG.parent / 'include'}",
]

# Files whose loops carry an MFMA accumulator through VALU code (the state walks' chunk-end update, the
# forward scan's per-head epilogue): with the default AGPR form the compiler copies the accumulator
# between AGPRs and VGPRs on every iteration (16 + 16 moves per 32 x 32 tile); the VGPR form keeps it in
# place. Not global: the other files are not measured with it.
MFMA_VGPR_FORM = {"ssd_state_fused.hip", "ssd_scan_fwd_fact.hip"}


def _run(cmd, verbose):
    if verbose:
        print(" ".join(str(c) for c in cmd), flush=True)
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(map(str, cmd))}\n{out}")
    if verbose and out.strip():
        print(out)


def _stale(src: Path, obj: Path) -> bool:
    """True when obj is missing or older than src or any header of csrc/ and include/."""
    if not obj.exists():
        return True
    deps = [src, *CSRC.glob("*.h"), *(PKG.parent / "include").glob("*.h")]
    return obj.stat().st_mtime < max(p.stat().st_mtime for p in deps)


def build(jobs: int = 8, verbose: bool = False, changed_only: bool = False) -> Path:
    """Compile csrc/*.hip and link the library. changed_only recompiles only objects older than their
    source or any header (a development shortcut; the default compiles everything)."""
    BUILD.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    objs = [BUILD / (s.stem + ".o") for s in sources]
    todo = [(s, o) for s, o in zip(sources, objs) if not changed_only or _stale(s, o)]

    def compile_one(pair):
        src, obj = pair
        extra = ["-mllvm", "-amdgpu-mfma-vgpr-form"] if src.name in MFMA_VGPR_FORM else []
        _run([HIPCC, *CFLAGS, *extra, "-c", str(src), "-o", str(obj)], verbose)

    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        list(ex.map(compile_one, todo))
    tmp = LIB.with_suffix(".so.tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)], verbose)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=min(8, os.cpu_count() or 1))
    ap.add_argument("--verbose", action="store_true")
    ap.add_argument("--changed", action="store_true", help="recompile only stale objects")
    a = ap.parse_args()
    path = build(a.jobs, a.verbose, a.changed)
    print(f"built {path}")
    sys.exit(0)
