"""Builds the native library libcasl_reinit.so in-tree for gfx950.

forest.cpp (host C++) is compiled with g++, the HIP sources with hipcc for
gfx950 only, and the objects are linked by hipcc into one shared library next
to this file.  The build always recompiles (it is the build check), and
writes objects under casl_p4est_amd/_build/.
"""
import os
import shutil
import subprocess
from concurrent.futures import ThreadPoolExecutor
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libcasl_reinit.so")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX_HOST", "g++")

HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    # strict IEEE evaluation: the FP64 path must reproduce the reference's
    # operation order exactly
    "-ffp-contract=off",
    # FP32 division/sqrt may be approximate: only the mixed path computes in
    # FP32 and its accuracy bar is relative to FP64 (1e-3 h); FP64 is unaffected
    "-fno-hip-fp32-correctly-rounded-divide-sqrt",
    # no packed FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the AMDGPU backend's instruction-level-parallelism scheduling strategy:
    # the stage kernels measured 0.9 % (FP32) and 0.5 % (FP64) faster with it,
    # at the same register counts and results
    "-mllvm", "-amdgpu-sched-strategy=max-ilp",
    # host functions and loops on cache lines: a network's He initialization
    # (51K normal deviates) takes 2.3 ms, and 3.8 where a change elsewhere moves
    # the generator's loop to the end of a line
    "-Xarch_host", "-falign-functions=64", "-Xarch_host", "-falign-loops=64",
    "-I", INCLUDE, "-I", CSRC,
]
HOST_FLAGS = ["-O2", "-fPIC", "-std=c++17", "-ffp-contract=off", "-pthread", "-I", INCLUDE, "-I", CSRC]

HIP_SOURCES = ["reinit.hip", "batch.hip", "mlp.hip", "curv.hip", "derivatives.hip", "advect.hip", "gpu_forest.hip",
               "curv_grid.hip", "noalloc.hip", "tiles_gpu.hip", "devmem.hip"]
HOST_SOURCES = ["forest.cpp", "tiles.cpp"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def build_library(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    jobs = []
    for src in HOST_SOURCES:
        obj = os.path.join(BUILD, src + ".o")
        jobs.append((obj, [CXX, *HOST_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]))
    for src in HIP_SOURCES:
        obj = os.path.join(BUILD, src + ".o")
        jobs.append((obj, [HIPCC, *HIP_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]))
    # one compiler per source, as many at once as there are cores
    workers = max(1, min(len(jobs), os.cpu_count() or 1, 8))
    with ThreadPoolExecutor(workers) as ex:
        list(ex.map(lambda job: _run(job[1], verbose), jobs))
    objs = [obj for obj, _ in jobs]
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-pthread"], verbose)
    os.replace(tmp, LIB)
    return LIB


def build_c_caller(verbose=True):
    """The test program that calls the library from C++ through
    include/casl_reinit.h alone (tests/c_abi), compiled with the host g++."""
    root = os.path.dirname(HERE)
    src = os.path.join(root, "tests", "c_abi", "reinit_caller.cpp")
    out = os.path.join(root, "tests", "c_abi", "reinit_caller")
    _run([CXX, "-O2", "-std=c++17", "-Wall", "-Wextra", "-I", INCLUDE, src, "-o", out, "-L", HERE, "-lcasl_reinit",
          "-Wl,-rpath,$ORIGIN/../../casl_p4est_amd"], verbose)
    return out


def build_oracle(verbose=True):
    oracle_dir = os.path.join(os.path.dirname(HERE), "oracle")
    _run(["make", "-s", "-C", oracle_dir], verbose)
    return os.path.join(oracle_dir, "liboracle.so")


if __name__ == "__main__":
    build_library(verbose=True)
    if "--oracle" in sys.argv:
        build_oracle(verbose=True)
