"""Builds the gfx950 CryoSPH library in-tree.

    python microgravity-cryogenic-multi-phase-sph-solver_amd/build.py [--jobs N]

Outputs (next to this file):
  libcryosph.so                         C ABI of include/cryosph.h (HIP kernels + host orchestration)
  CryoSPH.cpython-*.so                  Python module `CryoSPH` (pybind11 over the C ABI)

Every HIP translation unit is compiled for gfx950 only, with -ffp-contract=off
(no fused multiply-add: per-pair arithmetic rounds like the reference CPU
build) and with packed FP32 instructions disabled.
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent
CSRC = HERE / "csrc"
OBJ = HERE / "_build"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

LIB_SOURCES = ["kernels_forces_akinci.hip", "kernels_forces_csf.hip", "kernels_forces_none.hip", "kernels_grid.hip",
               "kernels_physics.hip", "kernels_step.hip", "kernels_adjoint.hip", "solver.cpp",
               "geometry.cpp", "io.cpp"]
COMMON = ["-O3", "-fPIC", "-std=c++17", "-ffp-contract=off", "-Wno-unknown-pragmas",
          f"-I{ROOT / 'include'}", f"-I{CSRC}"]
# -simplifycfg-sink-common=false: merging the identical tails of two branches
# (conditional accumulations in the pair loops) makes LLVM select between the
# accumulators' addresses, which forces them out of registers into scratch.
DEVICE = ["--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-fno-gpu-rdc", "-mllvm", "-simplifycfg-sink-common=false"]


def run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + r.stdout + r.stderr)
        raise SystemExit(f"build failed: {cmd[-1]}")
    return r


def compile_one(src: str) -> Path:
    out = OBJ / (src + ".o")
    srcp = CSRC / src
    # host sources (.cpp) go through the same HIP front end so that the shared
    # __host__ __device__ maths and the rounding flags are identical
    cmd = [HIPCC, *COMMON, *DEVICE, "-x", "hip", "-c", str(srcp), "-o", str(out)]
    run(cmd)
    return out


def build(jobs: int = 8, python_module: bool = True) -> None:
    OBJ.mkdir(exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(compile_one, LIB_SOURCES))
    lib = HERE / "libcryosph.so"
    tmp = HERE / "libcryosph.so.tmp"
    run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs),
         "-Wl,-soname,libcryosph.so"])
    os.replace(tmp, lib)
    if python_module:
        import pybind11
        suffix = sysconfig.get_config_var("EXT_SUFFIX")
        mod = HERE / f"CryoSPH{suffix}"
        tmpm = HERE / f"CryoSPH{suffix}.tmp"
        run(["g++", "-O2", "-fPIC", "-shared", "-std=c++17", f"-I{ROOT / 'include'}",
             f"-I{pybind11.get_include()}", f"-I{sysconfig.get_paths()['include']}",
             str(CSRC / "bindings.cpp"), "-o", str(tmpm), f"-L{HERE}", "-lcryosph", "-Wl,-rpath,$ORIGIN"])
        os.replace(tmpm, mod)


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=8)
    ap.add_argument("--no-python", action="store_true")
    a = ap.parse_args()
    build(a.jobs, not a.no_python)
    print("built", HERE / "libcryosph.so")
