"""Builds libevotrees_hip.so for gfx950 with hipcc (cross-compiles without a GPU)."""
import os
import platform
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libevotrees_hip.so")
SOURCES = ["api.hip", "kernels_data.hip", "kernels_grad.hip", "kernels_hist.hip", "kernels_scan.hip", "kernels_small.hip", "kernels_path.hip", "kernels_part.hip",
           "kernels_predict.hip", "predict_static.hip", "kernels_quantile.hip", "probes.hip", "pool.hip", "upload.hip", "model.hip", "host_bin.cpp", "host_bin_avx512.cpp"]
# -ffp-contract=off: the split gains follow the reference's expression order without fused multiply-add.
# packed-fp32 instructions are disabled for all device code.
# -amdgpu-kernarg-preload-count: a kernel's leading scalar and pointer arguments (up to 16 words) are in scalar registers when its wavefronts start; read from
# memory they are the first trip of every launch.  An empty-handed kernel of 256 blocks takes 1.56 us with it, 1.84 without; k_copy_words 2.46 -> 2.1.
FLAGS = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off", "-Xclang", "-target-feature", "-Xclang",
         "-packed-fp32-ops", "-mllvm", "-amdgpu-kernarg-preload-count=16", "-Wall", "-Wno-unused-result"]
# host-only sources; one of them is compiled for AVX-512 and called only on processors that have it
HOST_FLAGS = ["-x", "c++", "-O3", "-fPIC", "-std=c++17", "-ffp-contract=off", "-Wall"]
AVX512 = ["-mavx512f", "-mavx512bw", "-mavx512vl", "-mavx512dq"] if platform.machine() == "x86_64" else []


def _compile(src):
    obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
    flags = FLAGS if src.endswith(".hip") else HOST_FLAGS + (AVX512 if "avx512" in src else [])
    cmd = ["hipcc"] + flags + ["-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, res.stdout, res.stderr))
    return obj, res.stderr


def build(verbose=False):
    with ThreadPoolExecutor(max_workers=4) as ex:
        results = list(ex.map(_compile, SOURCES))
    objs = [r[0] for r in results]
    if verbose:
        for _, err in results:
            if err.strip():
                sys.stderr.write(err)
    cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-pthread", "-o", OUT] + objs
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (res.stdout, res.stderr))
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
