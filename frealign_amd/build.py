"""Build libfrealign_hip.so (gfx950) in-tree with hipcc.

python -m frealign_amd.build            # compile every source, link the library
"""
from __future__ import annotations

import os
import re
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

# compiled once more for each FFT length (fr_fft_dev.h): a code object per length
LENGTH_SOURCES = ["fr_prep.hip", "fr_cc3m_fft.hip", "fr_fft.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("FR_ARCH", "gfx950")
COMMON = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # no packed-FP32 instruction selection (v_pk_*_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def lengths() -> list[str]:
    with open(os.path.join(CSRC, "fr_fft_dev.h")) as f:
        macro = re.search(r"#define FR_LENGTHS\(X\)((?:.*\\\n)+.*\n)", f.read()).group(1)
    return re.findall(r"X\((\d+)\)", macro)


def _compile(job: tuple[str, str]) -> str:
    src, length = job
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ("_" + length if length else "") + ".o")
    path = os.path.join(CSRC, src)
    cmd = [HIPCC, *COMMON, *([f"-DFR_LEN={length}"] if length else []), "-c", path, "-o", obj]
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
    jobs = [(s, "") for s in srcs] + [(s, n) for s in LENGTH_SOURCES for n in lengths()]
    with ThreadPoolExecutor(max_workers=8) as ex:
        objs = list(ex.map(_compile, jobs))
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
