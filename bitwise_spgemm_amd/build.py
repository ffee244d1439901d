"""Build libbws.so in-tree with hipcc for gfx950.

Every translation unit under ``csrc/`` is compiled to an object in ``_build/``
(in parallel), then linked into ``bitwise_spgemm_amd/libbws.so``.  HIP code is
compiled with packed FP32 instructions disabled (``-packed-fp32-ops``).

Usage: ``python -m bitwise_spgemm_amd.build`` or ``build()`` from Python.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD_DIR = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libbws.so")
ARCH = "gfx950"

HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-pragmas",
    f"-I{INCLUDE}", f"-I{CSRC}",
]

# Per-file flags.  The SpMM MFMA kernels keep their accumulators in
# architectural VGPRs (the VGPR form of v_mfma): the wave tiles there need at
# most 128 accumulator registers, and the AGPR form makes the compiler copy
# accumulators between register files around the empty-stage branch.
FILE_FLAGS = {
    "spmm_mfma.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "spmm_direct16.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "spmm_direct.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    "spmm_planes.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"],
    # 128 x 128 wave tiles: 256 accumulators live in AGPRs
    "spmm_mfma_big.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=0"],
    "sddmm_mfma_big.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=0"],
}


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libbws.so)")


def sources():
    out = []
    for name in sorted(os.listdir(CSRC)):
        if name.endswith((".hip", ".cpp")):
            out.append(os.path.join(CSRC, name))
    return out


def _compile(src: str) -> str:
    obj = os.path.join(BUILD_DIR, os.path.basename(src) + ".o")
    cmd = [_hipcc()] + HIP_FLAGS + FILE_FLAGS.get(os.path.basename(src), []) + ["-c", src, "-o", obj]
    if src.endswith(".hip"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build(jobs: int | None = None, verbose: bool = False) -> str:
    """Compile every source and link libbws.so; returns the library path."""
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), max(1, (os.cpu_count() or 2)))
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
