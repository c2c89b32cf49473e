"""Compile libmiikv.so (HIP, gfx950) in-tree with hipcc.

The library is the product: C-ABI entry points declared in ``include/miikv.h``.
It is built here (cross-compiling works without a GPU) and the resulting
``miinfer_amd/libmiikv.so`` travels with the source tree to the GPU box.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libmiikv.so")
ARCH = "gfx950"

SOURCES = [
    "miikv_cache.hip",
    "miikv_decode.hip",
    "miikv_suffix.hip",
    "miikv_host.cpp",
    "miikv_session.cpp",
]

# Per-source code-generation options.  The suffix kernel keeps its MFMA
# accumulators in architectural VGPRs (see the note in miikv_suffix.hip).
SOURCE_FLAGS = {
    # Its step loops start on 64-byte boundaries: where they fall by chance moved config 4
    # by 1% (135.4 / 137.0 us).
    "miikv_suffix.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-falign-loops=64"],
    # The split-K decode kernels are scheduled for instruction-level parallelism
    # (config 2 at 32k: 20.2 -> 19.8 us per layer-token; config 3 unchanged; the
    # suffix kernel measured no better with it, so it keeps the default).
    "miikv_decode.hip": ["-mllvm", "--amdgpu-sched-strategy=max-ilp"],
}

FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    # Keep the compiler from forming packed fp32 ops (v_pk_*_f32).
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    return "hipcc"


def _run(cmd, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature; drop that noise.
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed ({res.returncode}):\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)


def build(verbose: bool = False) -> str:
    """Compile each source to an object (in parallel), then link libmiikv.so."""
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    compile_flags = [f for f in FLAGS if f != "-shared"]
    procs, objs = [], []
    for src in SOURCES:
        obj = os.path.join(objdir, src + ".o")
        objs.append(obj)
        cmd = [hipcc(), *compile_flags, *SOURCE_FLAGS.get(src, []), "-I", os.path.join(ROOT, "include"),
               "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.PIPE, text=True)))
    for cmd, p in procs:
        _, stderr = p.communicate()
        err = "\n".join(l for l in stderr.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed ({p.returncode}): {' '.join(cmd)}\n{err}")
    _run([hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", LIB + ".tmp", *objs], verbose)
    os.replace(LIB + ".tmp", LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
