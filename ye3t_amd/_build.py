"""Build the in-tree HIP library ``ye3t_amd/libye3t_hip.so`` for gfx950.

hipcc cross-compiles without a GPU, so this runs anywhere the ROCm toolchain
is installed.  Objects are compiled in parallel and linked into one shared
library exposing the C ABI of ``include/ye3t_hip.h``.
"""

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB = os.path.join(PKG, "libye3t_hip.so")
SOURCES = ("api.hip", "density.hip", "density_grad.hip", "density_grad_mfma.hip", "density_mfma.hip",
           "density_mfma64.hip", "density_species.hip", "factorized.hip", "monomial.hip", "neighbors.hip", "product.hip")
ARCH = os.environ.get("YE3T_HIP_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in ordinary VGPRs: no AGPR copies around each MFMA in
    # the branchy per-atom accumulation loops of the density kernels
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wno-unused-result", f"-I{INCLUDE}", f"-I{CSRC}",
]

# Flags of single sources.  density_grad_mfma.hip: the fp64 constants of its
# basis math stay where they are used; hoisted out of the loop over chunks they
# take 40 registers and push the kernels into scratch.
SOURCE_FLAGS = {"density_grad_mfma.hip": ["-mllvm", "-disable-machine-licm"]}


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def build_library(verbose=False):
    build_dir = os.path.join(ROOT, "_build")
    os.makedirs(build_dir, exist_ok=True)
    hipcc = _hipcc()

    def compile_one(src):
        obj = os.path.join(build_dir, src.replace(".hip", ".o"))
        cmd = [hipcc, *HIPCC_FLAGS, *SOURCE_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{res.stderr[-4000:]}")
        if verbose and res.stderr.strip():
            print(res.stderr, file=sys.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=len(SOURCES)) as pool:
        objs = list(pool.map(compile_one, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-lhiprtc"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr[-4000:]}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build_library(verbose=True))
