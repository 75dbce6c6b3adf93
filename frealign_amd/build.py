"""Build libfrealign_hip.so (gfx950) in-tree with hipcc.

python -m frealign_amd.build            # compile every source, link the library
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libfrealign_hip.so")
BUILD = os.path.join(HERE, "_build")

SOURCES = [
    "fr_api.cpp",
    "fr_host.cpp",
    "fr_fft.hip",
    "fr_prep.hip",
    "fr_extract.hip",
    "fr_cc3m.hip",
    "fr_cc3m_fft.hip",
    "fr_insert.hip",
    "fr_final.hip",
    "fr_stats.hip",
    "fr_search.hip",
    "fr_lists.hip",
    "fr_search_sep.hip",
    "fr_search_f32.hip",
    "fr_cnn.hip",
    "fr_cnn_train.hip",
    "fr_refine.cpp",
    "fr_sigma.hip",
    "fr_plan.cpp",
    "fr_fortran.cpp",
    "fr_ccp.hip",
    "fr_psearch.cpp",
    "fr_local.hip",
    "fr_ctfrefine.cpp",
    "fr_io.cpp",
    "fr_fpart.hip",
    "fr_finalize.cpp",
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FR_ARCH", "gfx950")
COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # no packed-FP32 instruction selection (v_pk_*_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    path = os.path.join(CSRC, src)
    cmd = [HIPCC, *COMMON, "-c", path, "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    return obj


def build(verbose: bool = True) -> str:
    if shutil.which(HIPCC) is None and not os.path.exists(HIPCC):
        raise RuntimeError(f"hipcc not found at {HIPCC}")
    os.makedirs(BUILD, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", f"--offload-arch={ARCH}", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    try:
        build()
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
