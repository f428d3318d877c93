"""Build libkrq.so (the gfx950 HIP kernels + C ABI) in-tree with hipcc.

    python kernel-rush-qwen_amd/build_lib.py

One hipcc -c per source (run in parallel), then one hipcc -shared link. Objects go to
kernel-rush-qwen_amd/_build/, the library to kernel-rush-qwen_amd/kernels/libkrq.so.

    python kernel-rush-qwen_amd/build_lib.py --timeline

builds the same sources with -DKRQ_TIMELINE (per-block wall-clock stamps in the FP8 GEMV, read by
timeline.py) into kernels/libkrq_timeline.so; the shipped library never carries them.
"""

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
OUT = os.path.join(HERE, "kernels", "libkrq.so")
TIMELINE_OUT = os.path.join(HERE, "kernels", "libkrq_timeline.so")
SOURCES = ["quant.hip", "gemv_fp8.hip", "gemv_bf16.hip", "lmhead.hip", "mlp.hip", "fused_gemv.hip", "fused_fp8.hip", "gemm_fp8.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# -packed-fp32-ops: no v_pk_{add,mul,fma}_f32 in the generated code.
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
# The row kernels (quantizers, RMSNorm rows) are one chain of dependent steps of about 0.5 us beside
# the launch itself, and its first link is the read of the kernel's arguments: these files have them
# preloaded into scalar registers (the first 16 words). Decode over 8 layers in one graph, same card:
# M = 16 302.5 -> 296.8 us, M = 5 296.6 -> 290.2, the fused layer at M = 16 347.9 -> 342.5. The GEMVs
# (weight streams, bound by HBM) measured the same with it and M = 1 0.3% slower, so they keep the load.
PRELOAD = ["-mllvm", "-amdgpu-kernarg-preload-count=16"]
FILE_FLAGS = {"quant.hip": PRELOAD, "fused_fp8.hip": PRELOAD}


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")


def build(verbose=False, timeline=False):
    build_dir = os.path.join(BUILD, "timeline") if timeline else BUILD
    out = TIMELINE_OUT if timeline else OUT
    flags = FLAGS + (["-DKRQ_TIMELINE"] if timeline else [])
    os.makedirs(build_dir, exist_ok=True)
    objs = [os.path.join(build_dir, src.replace(".hip", ".o")) for src in SOURCES]

    def compile_one(src, obj):
        cmd = [HIPCC, *flags, *FILE_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    workers = max(1, min(len(SOURCES), os.cpu_count() or 1))
    with ThreadPoolExecutor(max_workers=workers) as pool:
        list(pool.map(compile_one, SOURCES, objs))  # re-raises the first failure
    tmp = out + ".tmp"
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, out)
    return out


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv, timeline="--timeline" in sys.argv))
