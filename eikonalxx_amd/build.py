"""Builds libeikonalxx_amd.so (the HIP kernels and the C ABI) for gfx950.

Usage: python -m eikonalxx_amd.build [--verbose]

Every translation unit is compiled with -ffp-contract=off (the double
precision sweeps keep the reference's operation order, so they reproduce it
bit for bit), with -fno-honor-nans (no value of the solver is ever NaN: times
are finite or the 1e10 sentinel and square roots are taken of positive
arguments only, so fmin/fmax need no NaN-quieting of their operands -- one
canonicalising instruction per operand in IEEE mode) and with packed FP32
instructions disabled.
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libeikonalxx_amd.so")
SOURCES = ["ekx_kernels3d.hip", "ekx_flow3d.hip", "ekx_kernels2d.hip",
           "ekx_fields.hip", "ekx_model3d.hip", "ekx_capi.hip",
           "ekx_capi2d.hip"]
ARCH = os.environ.get("EKX_OFFLOAD_ARCH", "gfx950")


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def compile_flags():
    return ["--offload-arch=" + ARCH, "-O3", "-std=c++17", "-fPIC",
            "-ffp-contract=off", "-fno-honor-nans", "-fvisibility=hidden",
            "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
            "-Wall", "-Wno-unused-function",
            "-I" + os.path.join(ROOT, "include"), "-I" + CSRC]


# Per-source flags.  The column, flow and band kernels are scheduled for
# instruction-level parallelism: their steps are bound by VALU issue and
# dependency latency at a residency that LDS (3D) or the few waves of a
# problem (2D) fix, not by registers.
SOURCE_FLAGS = {
    "ekx_kernels3d.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"],
    "ekx_flow3d.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"],
    "ekx_kernels2d.hip": ["-mllvm", "-amdgpu-sched-strategy=max-ilp"],
}


def _compile(src, verbose):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = ([hipcc()] + compile_flags() + SOURCE_FLAGS.get(src, []) +
           ["-c", os.path.join(CSRC, src), "-o", obj])
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("compile of %s failed:\n%s\n%s"
                           % (src, r.stdout, r.stderr))
    if verbose and r.stderr.strip():
        print(r.stderr, flush=True)
    return obj


def build(verbose=False):
    """Compiles every source and links the shared library (always)."""
    os.makedirs(BUILD, exist_ok=True)
    with concurrent.futures.ThreadPoolExecutor(max_workers=4) as ex:
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp]
    cmd += objs
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (r.stdout, r.stderr))
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="--verbose" in sys.argv))
