"""Build libshady_hip.so (all HIP sources, gfx950) in-tree with hipcc.

Usage: python -m shady_thinker_amd.build   (or build() from Python).
The library is a plain C-ABI shared object (include/shady_hip.h); it links
only the HIP runtime, not torch.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libshady_hip.so")
SOURCES = [
    "runtime.hip", "qmv.hip", "qmv_i4_p0.hip", "qmv_i4_p1.hip", "qmv_i4t_p0.hip", "qmv_i4t_p1.hip", "qmv_i8.hip", "qmv_i8t.hip",
    "i8mm.hip", "i4mm.hip", "i4xs.hip", "i4xs_f32.hip", "i4xs_f32d.hip", "i4xs_f32s.hip", "i4xs_f16.hip", "i4xs_f16d.hip",
    "i4xs_f16g.hip", "dequant.hip", "gemm.hip", "bf16mv.hip",
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    # Packed-FP32 VALU forms are kept out of every kernel (some of their forms
    # have given wrong results on this hardware).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
    "-I", CSRC,
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    # hipcc's host pass warns that it does not know the packed-fp32 feature;
    # that is expected, everything else is shown.
    warn = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if warn:
        print(f"[{src}] {warn}", file=sys.stderr)
    return obj


def build(verbose: bool = True) -> str:
    """Compile every HIP source (always) and link libshady_hip.so."""
    os.makedirs(OBJ, exist_ok=True)
    missing = [s for s in SOURCES if not os.path.exists(os.path.join(CSRC, s))]
    if missing:
        raise RuntimeError(f"listed in SOURCES, not in {CSRC}: {' '.join(missing)}")
    with cf.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    # (a symbol that no source defines fails here, not when the library is loaded)
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,--no-undefined", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build()
