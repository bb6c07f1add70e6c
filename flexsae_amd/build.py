"""Builds libflexsae_amd.so (the C-ABI library of HIP kernels) with hipcc for gfx950 and _eager.so (the extension module that
calls it for ordinary eager calls, over torch's C++ interface) with g++, both in-tree.

Usage: python -m flexsae_amd.build
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_PATH = os.path.join(HERE, "libflexsae_amd.so")
EAGER_PATH = os.path.join(HERE, "_eager.so")

# gfx950 only: some kernels use more LDS per workgroup than the 64 KiB of earlier gfx9 parts
# (csr_sort_long_kernel 65 600 bytes, the hot-latent variant of the training-step kernel more), the
# gfx950 lane-swap and bf16 conversion instructions, and buffer loads with the LDS as destination.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-shared",
    "-munsafe-fp-atomics",
    # keep the compiler from forming packed-fp32 instructions out of scalar float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
]
# (the macros are what torch's own headers ask for)
EAGER_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1"]


def source_id(extra_flags=()) -> str:
    """Identifier of what the library and the extension module are built from: a hash over the sources of
    both, the header and the compiler flags (not over the binaries, so that rebuilding the same sources gives
    the same id).  The library reports it through flexsae_build_id() and the module as its `build_id`, which have
    to agree; measurements kept under profiles/ carry it."""
    import hashlib

    h = hashlib.sha256()
    files = sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".hpp", ".cpp")))
    files.append(os.path.join(os.path.dirname(HERE), "include", "flexsae_amd.h"))
    for path in files:
        h.update(os.path.basename(path).encode())
        with open(path, "rb") as fh:
            h.update(fh.read())
    h.update(" ".join([*HIPCC_FLAGS, *extra_flags, *EAGER_FLAGS]).encode())
    return h.hexdigest()[:16]


def build_eager(verbose: bool = False, extra_flags=()) -> str:
    """``extra_flags``: those of the library it goes with, for its identifier."""
    import sysconfig

    import torch

    base = os.path.dirname(torch.__file__)
    include = [os.path.join(base, "include"), os.path.join(base, "include", "torch", "csrc", "api", "include"),
               os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    # (the libraries are loaded by torch, found by name)
    cmd = [os.environ.get("CXX", "g++"), *EAGER_FLAGS, f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DFLEXSAE_BUILD_ID="{source_id(extra_flags)}"', f'-DFLEXSAE_TORCH_VERSION="{torch.__version__}"',
           *(f"-isystem{d}" for d in include), os.path.join(CSRC, "eager.cpp"), "-o", EAGER_PATH,
           "-L" + os.path.join(base, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-ltorch"]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError("g++ failed building _eager.so")
    if verbose and proc.stderr:
        sys.stderr.write(proc.stderr)
    return EAGER_PATH


def build(verbose: bool = False, extra_flags=()) -> str:
    build_eager(verbose, extra_flags)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    cmd = [hipcc, *HIPCC_FLAGS, *extra_flags, f'-DFLEXSAE_BUILD_ID="{source_id(extra_flags)}"', "-o", LIB_PATH,
           os.path.join(CSRC, "flexsae_amd.hip")]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError("hipcc failed building libflexsae_amd.so")
    if verbose and proc.stderr:
        sys.stderr.write(proc.stderr)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
