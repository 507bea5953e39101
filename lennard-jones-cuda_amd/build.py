"""Build recipe of libljhip.so (gfx950) and of the test-oracle libraries.

    python lennard-jones-cuda_amd/build.py            # product + test oracles
    python lennard-jones-cuda_amd/build.py --product  # libljhip.so only

Outputs (in-tree, git-ignored, shipped with the tree to the GPU host):
    lennard-jones-cuda_amd/lib/libljhip.so
    lennard-jones-cuda_amd/lib/run_isotherm, run_fluctuations (task programs)
    oracle/liboracle.so, oracle/_ref/*.so  (test oracles; _ref only where the
                                            reference sources are present)
"""
import argparse
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB = os.path.join(PKG, "lib")
BUILD = os.path.join(PKG, "_build")
INCLUDE = os.path.join(ROOT, "include")
ORACLE = os.path.join(ROOT, "oracle")
REFERENCE = "/root/reference"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
# Packed FP32 (v_pk_*_f32) stays disabled: the j-loop is written for scalar
# FP32 issue and the packed forms are not used on this target.
HIPFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result", "-Wno-unknown-pragmas",
    f"-I{INCLUDE}", f"-I{CSRC}",
]

SOURCES = ["lj_kernels.hip", "lj_force_n3.hip", "lj_batch.hip", "lj_adjoint.hip", "lj_fp64.hip",
           "lj_noalloc.hip", "lj_fluct.hip", "lj_rdf_cells.hip", "lj_small.hip", "lj_host.cpp",
           "lj_api.cpp", "lj_batch_api.cpp", "lj_adjoint_api.cpp", "lj_fluct_api.cpp"]


def _run(cmd, cwd=None):
    r = subprocess.run(cmd, cwd=cwd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in r.stdout.splitlines()
                    if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{out}")
    return out


def build_product(verbose=False):
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIB, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]

    def compile_one(src):
        obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
        lang = ["-x", "hip"]
        out = _run([HIPCC, *HIPFLAGS, *lang, "-c", os.path.join(CSRC, src), "-o", obj])
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(compile_one, srcs))
    target = os.path.join(LIB, "libljhip.so")
    tmp = target + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, target)
    return target


def build_driver():
    """The C++ program that drives the header-only MDSystem class over the
    C-ABI (include/lj_mdsystem.hpp); run by the GPU tests."""
    src = os.path.join(ROOT, "tests", "cpp", "mdsystem_driver.cpp")
    out = os.path.join(LIB, "mdsystem_driver")
    _run(["g++", "-std=c++11", "-O2", "-Wall", "-Wextra", "-Werror", f"-I{INCLUDE}", src,
          f"-L{LIB}", "-lljhip", "-Wl,-rpath,$ORIGIN", "-o", out + ".tmp"])
    os.replace(out + ".tmp", out)
    return out


TASKS = ["run_isotherm", "run_fluctuations"]


def build_tasks():
    """The task programs (the reference's src/tasks drivers over the C-ABI)."""
    out = []
    for name in TASKS:
        src = os.path.join(PKG, "tasks", name + ".cpp")
        exe = os.path.join(LIB, name)
        _run(["g++", "-std=c++11", "-O2", "-Wall", "-Wextra", "-Werror", f"-I{INCLUDE}",
              f"-I{os.path.join(PKG, 'tasks')}", src, f"-L{LIB}", "-lljhip",
              "-Wl,-rpath,$ORIGIN", "-o", exe + ".tmp"])
        os.replace(exe + ".tmp", exe)
        out.append(exe)
    return out


def build_valu_rates():
    """The issue-rate measurement program (csrc/valu_rates.hip)."""
    exe = os.path.join(LIB, "valu_rates")
    _run([HIPCC, *HIPFLAGS, "-x", "hip", os.path.join(CSRC, "valu_rates.hip"), "-o", exe + ".tmp"])
    os.replace(exe + ".tmp", exe)
    return exe


def build_oracles():
    _run(["make", "-s", "-C", ORACLE, "oracle"])
    if os.path.isdir(os.path.join(REFERENCE, "src", "library")):
        _run(["make", "-s", "-C", ORACLE, "ref", f"REF={REFERENCE}"])


def build_all(product_only=False, verbose=False):
    t = build_product(verbose=verbose)
    build_driver()
    build_tasks()
    build_valu_rates()
    if not product_only:
        build_oracles()
    return t


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--product", action="store_true", help="build libljhip.so only")
    ap.add_argument("-v", action="store_true")
    a = ap.parse_args()
    print(build_all(product_only=a.product, verbose=a.v))
