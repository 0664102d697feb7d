"""Build libp4gpu.so (HIP kernels + C-ABI) for gfx950, in-tree.

    python p4-phylogenetics_amd/build.py          # build the library
    python p4-phylogenetics_amd/build.py --clean  # remove build outputs

The shared library is written next to the Python package
(p4-phylogenetics_amd/p4gpu/libp4gpu.so) so that the package finds it
without any install step and it travels with the source tree.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "p4gpu")
LIB = os.path.join(OUT_DIR, "libp4gpu.so")
OBJ_DIR = os.path.join(HERE, "_build")
SOURCES = ["p4g_gamma.hip", "p4g_kernels.hip", "p4g_aa.hip", "p4g_api.hip", "p4g_mlp.hip", "p4g_deriv.hip", "p4g_anc.hip", "p4g_sim.hip", "p4g_compress.hip"]
ARCH = os.environ.get("P4G_OFFLOAD_ARCH", "gfx950")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    # keep the compiler from forming packed FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]


def _compile(src):
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns about the GPU-only target feature; drop that line
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    return obj


def build(verbose=True):
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with ThreadPoolExecutor(max_workers=min(4, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


def clean():
    for f in [LIB]:
        if os.path.exists(f):
            os.remove(f)
    if os.path.isdir(OBJ_DIR):
        for f in os.listdir(OBJ_DIR):
            os.remove(os.path.join(OBJ_DIR, f))


if __name__ == "__main__":
    if "--clean" in sys.argv:
        clean()
    else:
        build()
