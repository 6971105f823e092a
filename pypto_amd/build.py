"""Builds the native parts in-tree: the C-ABI library with the gfx950 kernels and the pybind11
module on top of it.  ``python -m pypto_amd.build`` or :func:`build_all`."""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB_NAME = "libpypto_amd_sfa.so"
LIB_PATH = os.path.join(HERE, LIB_NAME)
EXT_PATH = os.path.join(HERE, "_C" + (sysconfig.get_config_var("EXT_SUFFIX") or ".so"))

HIP_SOURCES = ["sfa_kernels.hip", "li_kernels.hip", "lip_kernels.hip", "mlap_kernels.hip", "prolog_fused.hip", "capi.cpp"]
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # fuse a*b+c only where the source writes it in one expression; files that need exact
    # multiply-then-add semantics switch it off with a pragma (the default, "fast", ignores pragmas)
    "-ffp-contract=on",
    # packed fp32 arithmetic is switched off for all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-inline-asm",
]


def _run(cmd):
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    lines = [ln for ln in res.stdout.splitlines() if "is not a recognized feature for this target" not in ln]
    if res.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(cmd) + "\n" + "\n".join(lines))
    return "\n".join(lines)


def build_library(verbose: bool = False) -> str:
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc] + HIPCC_FLAGS + ["-x", "hip", "-I" + INCLUDE, "-I" + CSRC] + \
          [os.path.join(CSRC, s) for s in HIP_SOURCES] + ["-o", LIB_PATH]
    out = _run(cmd)
    if verbose and out:
        print(out)
    return LIB_PATH


def build_extension(verbose: bool = False) -> str:
    import pybind11
    import torch
    cxx = os.environ.get("CXX", "g++")
    torch_dir = os.path.dirname(os.path.abspath(torch.__file__))
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    # torch_calls.cpp reads torch tensors directly; torch's libraries are in the process before this module is loaded
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           "-I" + INCLUDE, "-I" + pybind11.get_include(), "-I" + sysconfig.get_paths()["include"],
           "-isystem", os.path.join(torch_dir, "include"),
           "-isystem", os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(rocm, "include"),
           os.path.join(CSRC, "pybind.cpp"), os.path.join(CSRC, "torch_calls.cpp"), "-o", EXT_PATH,
           "-L" + HERE, "-l:" + LIB_NAME, "-Wl,-rpath,$ORIGIN",
           "-L" + os.path.join(torch_dir, "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    out = _run(cmd)
    if verbose and out:
        print(out)
    return EXT_PATH


def build_all(verbose: bool = False):
    return build_library(verbose), build_extension(verbose)


if __name__ == "__main__":
    for path in build_all(verbose=True):
        print("built", path)
    sys.exit(0)
