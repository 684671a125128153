"""Build the native libraries in-tree (no JIT cache, so they travel with the
source tree):

* cable_amd/libcable_gpu.so  -- HIP kernels and C ABI (include/cable_gpu.h),
  compiled for gfx950 with hipcc;
* tests/libgpu_quotient.so -- a test's kernel (tests/gpu_quotient.hip);
* oracle/liboracle.so, oracle/_ref/*  -- the test oracle and, when the
  reference tree is present, the compiled reference (oracle/Makefile).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(ROOT, "cable_amd", "csrc")
LIB = os.path.join(ROOT, "cable_amd", "libcable_gpu.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    # no packed FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]
# per translation unit: the plain FP64 path reproduces the reference's
# rounding (no FMA contraction; the step's quotients and roots are
# cbm_physics.h's, IEEE's bits by shorter sequences); the mixed
# path is held to its flux tolerance and may contract within an expression
# and use the hardware approximations of the elementary functions
TU_FLAGS = {
    "cable_gpu.hip": ["-ffp-contract=off"],
    "cbm_kernels_fp64.hip": ["-ffp-contract=off"],
    # the mixed kernels also schedule for instruction-level parallelism
    # (measured 1.7% faster at two waves per SIMD; the FP64 kernels, at one
    # wave per SIMD, measured slower with it) and flush FP32 denormals, which
    # drops the range handling of the hardware exp/log sequences (3% of the
    # step's instructions; 2.7% faster at 1,048,576 tiles, same pass count).
    # They assume finite values and ignore the sign of zero (no NaN or
    # infinity arises in a valid step): the step's MIN/MAX selects become
    # single min/max instructions, and the static instruction count of the
    # step falls 11% (10% faster, the same flux statistics).  Reassociation
    # was also tried: it made the kernel instantiations (plain, capture,
    # hybrid) differ in their bits where they run the same method.
    "cbm_kernels_mixed.hip": ["-ffp-contract=on", "-fapprox-func", "-fgpu-flush-denormals-to-zero",
                              "-fno-honor-nans", "-fno-signed-zeros", "-fno-honor-infinities",
                              "-Xarch_device", "-mllvm=-misched=gcn-max-ilp"],
    "mlp.hip": ["-ffp-contract=on"],
}
# the resident plain step loops over a run's steps; hoisting a step's constants
# out of that loop would hold them in registers, and then in scratch memory,
# through every step (a day of 262,144 tiles in FP64 14.4 against 13.1 ms, of
# 1,048,576 in mixed precision 20.0 against 16.9 ms)
NO_HOIST = ["-Xarch_device", "-mllvm=-disable-machine-licm"]
# (and the FP64 step's one wave per SIMD gains from a schedule for
# instruction-level parallelism here: 13.0 -> 12.7 ms)
TU_FLAGS["cbm_run_fp64.hip"] = TU_FLAGS["cbm_kernels_fp64.hip"] + NO_HOIST + [
    "-Xarch_device", "-mllvm=-misched=gcn-iterative-ilp"]
TU_FLAGS["cbm_run_mixed.hip"] = TU_FLAGS["cbm_kernels_mixed.hip"] + NO_HOIST
# the FP64 drop-in step, whose per-tile parameters fill the registers, gains
# too (262,144 tiles 0.70 -> 0.68 ms); the hybrid kernels do not
TU_FLAGS["cbm_kernels_fp64.hip"] = TU_FLAGS["cbm_kernels_fp64.hip"] + NO_HOIST


def hipcc():
    for c in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def build_gpu(verbose=False):
    objdir = os.path.join(ROOT, "cable_amd", "_build")
    os.makedirs(objdir, exist_ok=True)
    import concurrent.futures as cf
    objs, cmds = [], []
    for src, extra in TU_FLAGS.items():
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmds.append((src, [hipcc()] + HIPCC_FLAGS + extra + ["-c", "-o", obj, os.path.join(CSRC, src)]))
        objs.append(obj)
    # the translation units compile independently: one process each
    with cf.ThreadPoolExecutor(max(1, min(len(cmds), os.cpu_count() or 1))) as ex:
        results = list(ex.map(lambda c: (c[0], subprocess.run(c[1], capture_output=True, text=True)), cmds))
    for src, r in results:
        if r.returncode != 0:
            sys.stderr.write(r.stdout + r.stderr)
            raise RuntimeError(f"hipcc failed for {src}")
    tmp = LIB + ".tmp"
    r = subprocess.run([hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs,
                       capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link failed for libcable_gpu.so")
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


def build_test_kernels(verbose=False):
    """tests/libgpu_quotient.so: the FP64 step's quotients and roots on host
    operands, with the flags of the FP64 kernels."""
    out = os.path.join(ROOT, "tests", "libgpu_quotient.so")
    r = subprocess.run([hipcc()] + HIPCC_FLAGS + TU_FLAGS["cbm_run_fp64.hip"] +
                       ["-shared", "-o", out + ".tmp", os.path.join(ROOT, "tests", "gpu_quotient.hip")],
                       capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stderr)
        raise RuntimeError("hipcc failed for tests/gpu_quotient.hip")
    os.replace(out + ".tmp", out)
    if verbose:
        print("built", out)


def build_oracle(with_reference=True, verbose=False):
    targets = ["oracle"]
    if with_reference and os.path.isdir("/root/reference/src"):
        # the compiled reference, and the reference driven through the
        # Fortran drop-in for cbm (needs libcable_gpu.so built first)
        targets += ["r8", "r4", "gpu8", "gpu4"]
    r = subprocess.run(["make", "-s", "-C", os.path.join(ROOT, "oracle")] + targets,
                       capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout[-4000:] + r.stderr[-4000:])
        raise RuntimeError("oracle build failed")
    if verbose:
        print("built oracle targets:", " ".join(targets))


def build_all(verbose=True):
    build_gpu(verbose)
    build_test_kernels(verbose)
    build_oracle(verbose=verbose)


if __name__ == "__main__":
    build_all()
