"""Builds libfpq_hip.so (the C-ABI HIP library, gfx950, hipcc) and _fpq_host.so (host code, g++), in-tree.

Usage: python fp-quant_amd/build.py [--force]
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "fp_quant", "_lib")
LIB = os.path.join(OUT_DIR, "libfpq_hip.so")
HOST = os.path.join(OUT_DIR, "_fpq_host.so")   # the native host path of the eager layers (an extension module)
SOURCES = ["fpq_capi.hip", "fpq_quantize.hip", "fpq_gemm.hip", "fpq_gemm_packed.hip", "fpq_gemm_stream.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt", "-fno-gpu-flush-denormals-to-zero",
    # packed fp32 VALU forms are not to be emitted on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def host_command():
    """Host code only: g++ against the headers and libraries of the installed PyTorch."""
    import sysconfig

    import torch

    root = os.path.dirname(torch.__file__)
    includes = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
                os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
            "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            *(f for d in includes for f in ("-isystem", d)), os.path.join(CSRC, "fpq_host.cpp"), "-o", HOST,
            "-L" + os.path.join(root, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python"]


def build(force: bool = True, verbose: bool = True) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    deps = [os.path.join(CSRC, f) for f in os.listdir(CSRC)] + [os.path.join(HERE, "..", "include", "fpq.h")]
    if not force and all(os.path.exists(out) and all(os.path.getmtime(d) <= os.path.getmtime(out) for d in deps)
                         for out in (LIB, HOST)):
        return LIB
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objs = []
    procs = []
    for src in SOURCES:
        obj = os.path.join(OUT_DIR, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [hipcc, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((cmd, subprocess.Popen(cmd)))
    host_cmd = host_command()
    if verbose:
        print(" ".join(host_cmd), flush=True)
    procs.append((host_cmd, subprocess.Popen(host_cmd)))
    for cmd, p in procs:
        if p.wait() != 0:
            raise RuntimeError("compiler failed: " + " ".join(cmd))
    link = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB]
    if verbose:
        print(" ".join(link), flush=True)
    subprocess.check_call(link)
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv or True))
