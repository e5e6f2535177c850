"""Builds kvmix_amd/libkvmix_hip.so (hand-written HIP kernels, gfx950 only) with hipcc."""
from __future__ import annotations

import os
import shutil
import subprocess
import sysconfig
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libkvmix_hip.so")
SOURCES = ["abi.hip", "quant_pack.hip", "dequant_gemv.hip", "decode_attn.hip", "fused_attn.hip", "linear_rows.hip", "prefill_attn.hip", "copy_rows.hip", "rope_append.hip", "stream_probe.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-fast-math",
    # packed fp32 instructions are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


HOST_SOURCE = os.path.join(CSRC, "host.cpp")
HOST_LIB = os.path.join(HERE, "_host.so")


def host_command() -> list:
    """The operators' host side: plain C++ against torch's headers, an extension module next to the library."""
    import torch
    from torch.utils import cpp_extension

    rocm = os.path.dirname(os.path.dirname(os.path.realpath(shutil.which("hipcc") or "/opt/rocm/bin/hipcc")))
    includes = cpp_extension.include_paths() + [os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    return [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}"] + [
            a for i in includes for a in ("-isystem", i)] + [HOST_SOURCE, "-o", HOST_LIB] + [
            "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"]


def build(verbose: bool = False) -> str:
    """Compiles every source (in parallel: one of them takes as long as all the others), links the library and builds
    the operators' host side."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, s + ".o") for s in SOURCES]

        commands = [[hipcc] + HIPCC_FLAGS + ["-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(SOURCES, objects)]

        def run(cmd):
            if verbose:
                print(" ".join(cmd), flush=True)
            subprocess.check_call(cmd)

        with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
            list(pool.map(run, [host_command()] + commands))
        subprocess.check_call([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objects + ["-o", LIB])
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
