"""Builds libqlora_hip.so (the C-ABI library) for gfx950 with hipcc.

Every translation unit is compiled in parallel into ``_build/`` and linked
in-tree next to the Python binding, so the library travels with the source
tree.  Usage: ``python vkqlora.rs_amd/build_lib.py`` (always rebuilds).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "qlora_hip", "libqlora_hip.so")
# measurement kernels for bench.py (a library of their own)
PROBE_SRC = "k_probe.hip"
PROBE_OUT = os.path.join(HERE, "qlora_hip", "libqh_probe.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

SOURCES = ["runtime.cpp", "nf4_file.cpp", "k_quant.hip", "k_gemm.hip", "k_gemm_bf16.hip",
           "k_gemv.hip",
           "k_dstream.hip", "k_dsplit.hip", "k_adam.hip", "k_elem.hip",
           "k_block.hip", "k_rank.hip", "k_slim.hip", "k_plane.hip"]

COMMON = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-fvisibility=hidden", "-ffp-contract=off",
    # packed fp32 VALU ops stay disabled on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"), "-I", CSRC,
    "-Wall", "-Wno-unused-result",
]


# Per-file flags: the decode stream kernel's step loop (8 steps per K-line,
# up to 48 steps) must unroll fully, past the default pragma size limit, so
# that its per-line register arrays stay in registers; its leading scalar
# arguments are preloaded into SGPRs.
EXTRA = {"k_dstream.hip": ["-mllvm", "-pragma-unroll-threshold=100000",
                           "-mllvm", "-amdgpu-kernarg-preload-count=16"],
         "k_dsplit.hip": ["-mllvm", "-pragma-unroll-threshold=100000"],
         "k_slim.hip": ["-mllvm", "-pragma-unroll-threshold=100000"]}


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, src + ".o")
    cmd = [HIPCC, *COMMON, *EXTRA.get(src, [])]
    if src.endswith(".cpp"):
        cmd += ["-x", "hip"]
    cmd += ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return obj


def _link(objs, out):
    tmp = out + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, out)


def build(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs = SOURCES + [PROBE_SRC]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = dict(zip(srcs, ex.map(_compile, srcs)))
    _link([objs[s] for s in SOURCES], OUT)
    _link([objs[PROBE_SRC]], PROBE_OUT)
    if verbose:
        print(f"built {OUT} and {PROBE_OUT}")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
