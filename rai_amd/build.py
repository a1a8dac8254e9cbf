"""Build librai_hip.so (gfx950) in-tree with hipcc.

Every source under rai_amd/csrc is compiled with FP contraction off (the
kernels fuse a multiply-add only where the reference uses an FMA intrinsic)
and with packed FP32 instructions disabled for device code.
"""
from __future__ import annotations

import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_obj")
LIB_DIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIB_DIR, "librai_hip.so")
RUN = os.path.join(LIB_DIR, "rai-run")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

COMMON = ["-O3", "-std=c++17", "-fPIC", "-ffp-contract=off", "-Wall",
          "-I", os.path.join(ROOT, "include"), "-I", CSRC]
DEVICE = [f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
SOURCES = ["kernels.hip", "fused.hip", "attn_mm.hip", "gemv.hip", "gemv_stream.hip", "gemm_mm.hip", "moe.hip", "sample.hip", "decode_gemv.hip", "tied_head.hip", "runtime.hip", "format.cpp", "synth.cpp"]
# Per-source device flags: the matrix-core GEMV keeps MFMA results in
# architectural VGPRs, which its epilogue reads directly (without it the
# compiler routes them through AGPRs and one copy per value).
EXTRA = {"gemv.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"], "gemm_mm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
         "gemv_stream.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
         "attn_mm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"]}


def _compile(src: str) -> str:
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJ, src + ".o")
    cmd = [HIPCC] + COMMON
    if src.endswith(".hip"):
        cmd += DEVICE + EXTRA.get(src, []) + ["-x", "hip"]
    cmd += ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass of hipcc does not know the packed-fp32 feature and says so;
    # that note is harmless and filtered out.
    noise = "is not a recognized feature for this target"
    msg = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{msg}")
    if msg.strip():
        print(msg, file=sys.stderr)
    return obj


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    # rai-run: the generate loop over the C ABI (host code only).
    run_tmp = RUN + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-I", os.path.join(ROOT, "include"), os.path.join(CSRC, "rai_run.cpp"),
           "-L", LIB_DIR, "-lrai_hip", "-Wl,-rpath,$ORIGIN", "-o", run_tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("rai-run build failed:\n" + r.stdout + r.stderr)
    os.replace(run_tmp, RUN)
    if verbose:
        print("built", LIB, "and", RUN)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
