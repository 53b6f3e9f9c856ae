"""Compile the gfx950 kernels, in-tree, next to the sources:

    libatorch_amd_fp8.so      the product library (include/atorch_amd_fp8.h)
    ../_host.so               the host side in native code (host.cpp), a Python extension module over the product library
    libatorch_amd_probes.so   measurement aids for the benchmark and the tests (include/atorch_amd_probes.h):
                              probes, and the grouped GEMMs with their launch choices pinned per call

    python -m atorch_amd.csrc.build          # or: python atorch_amd/csrc/build.py

hipcc cross-compiles for gfx950 without a GPU present.  Packed-FP32 instruction selection is
switched off for all device code.  Symbols other than the C entry points stay local to each library.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
SOURCES = ["capi.hip", "quant.hip", "permute.hip", "gemm.hip", "gemm_rows.hip", "gemm_rows_higher.hip", "gemm_wgrad.hip", "gemm_few.hip"]
PROBE_SOURCES = ["capi.hip", "gemm.hip", "gemm_rows.hip", "gemm_rows_higher.hip", "gemm_wgrad.hip", "gemm_few.hip", "probe.hip"]  # compiled with -DAAMD_TUNING
LIB = os.path.join(HERE, "libatorch_amd_fp8.so")
HOST = os.path.join(os.path.dirname(HERE), "_host.so")
PROBES_LIB = os.path.join(HERE, "libatorch_amd_probes.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fvisibility=hidden",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]  # fmt: skip
SOURCE_FLAGS = {"gemm_rows_higher.hip": ["-falign-loops=64"]}  # (what it is for stands there)
LINK = ["--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-Bsymbolic"]


def _build_host() -> None:
    """The Python extension module: host code only, compiled with g++ against torch's headers."""
    import sysconfig

    import torch

    t = os.path.join(os.path.dirname(torch.__file__))
    inc = [os.path.join(t, "include"), os.path.join(t, "include", "torch", "csrc", "api", "include"), "/opt/rocm/include",
           sysconfig.get_paths()["include"]]  # fmt: skip
    subprocess.check_call(
        [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-w",
         "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
         *[f"-I{d}" for d in inc], os.path.join(HERE, "host.cpp"), "-o", HOST,
         f"-L{os.path.join(t, 'lib')}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip",
         f"-L{HERE}", "-l:" + os.path.basename(LIB), "-Wl,-rpath,$ORIGIN/csrc"]
    )  # fmt: skip


def _compile(job) -> str:
    src, suffix, extra = job
    obj = os.path.join(HERE, src.replace(".hip", suffix + ".o"))
    subprocess.check_call([HIPCC, *FLAGS, *SOURCE_FLAGS.get(src, []), *extra, "-c", os.path.join(HERE, src), "-o", obj])
    return obj


def build(verbose: bool = False, extra_flags=()) -> str:
    extra = list(extra_flags)
    jobs = [(s, "", extra) for s in SOURCES] + [(s, ".probes", extra + ["-DAAMD_TUNING"]) for s in PROBE_SOURCES]
    with ThreadPoolExecutor(max_workers=8) as ex:
        objs = list(ex.map(_compile, jobs))
    subprocess.check_call([HIPCC, *LINK, "-o", LIB, *objs[: len(SOURCES)]])
    subprocess.check_call([HIPCC, *LINK, "-o", PROBES_LIB, *objs[len(SOURCES) :]])
    _build_host()
    if verbose:
        print("built", LIB)
        print("built", PROBES_LIB)
        print("built", HOST)
    return LIB


if __name__ == "__main__":
    build(verbose=True, extra_flags=sys.argv[1:])
