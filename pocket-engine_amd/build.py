"""Builds, in-tree next to the Python package that loads them:
- libpkv.so: HIP kernels for gfx950 + the C-ABI + the host KV manager;
- pkv_kernels.hsaco: the same kernel bodies under the reference engine's
  kernel names and signatures (a code object for hipModuleLoadData)."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "pkv", "libpkv.so")
HSACO = os.path.join(HERE, "pkv", "pkv_kernels.hsaco")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# Packed FP32 instructions are kept out of every code object.
COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]
# MFMA results in whatever registers hold them: without it the compiler keeps
# the accumulators of a kernel that may use more than 256 registers in the
# accumulation half throughout, and copies each out and back around every
# rescale (1,424 copies in verify_range_kernel<6, 4>, 76 with it; no other
# kernel of the library changes). 24 x 4 draft rows at 12 / 2 heads, 900 to
# 16,000 keys, 115.0 -> 106.1 us; 4 x 4 over 500 keys 17.1 -> 16.1.
FLAGS = COMMON + ["-fPIC", "-shared", "-mllvm", "-amdgpu-mfma-vgpr-form"]
SOURCES = ["pkv_capi.hip", "pkv_host.cpp"]


def _run(cmd, what, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"{what} build failed")


def build(verbose=False):
    _run([HIPCC] + FLAGS + [os.path.join(CSRC, s) for s in SOURCES] + ["-o", OUT], "libpkv.so", verbose)
    _run([HIPCC, "--genco"] + COMMON + [os.path.join(CSRC, "pkv_refabi.hip"), "-o", HSACO], "pkv_kernels.hsaco",
         verbose)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
