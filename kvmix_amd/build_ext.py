"""Builds kvmix_amd/libkvmix_hip.so (hand-written HIP kernels, gfx950 only) with hipcc."""
from __future__ import annotations

import os
import shutil
import subprocess
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libkvmix_hip.so")
SOURCES = ["abi.hip", "quant_pack.hip", "dequant_gemv.hip", "decode_attn.hip", "fused_attn.hip", "linear_rows.hip", "prefill_attn.hip", "rope_append.hip", "stream_probe.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-fast-math",
    # packed fp32 instructions are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def build(verbose: bool = False) -> str:
    """Compiles every source (in parallel: one of them takes as long as all the others) and links the library."""
    hipcc = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    with tempfile.TemporaryDirectory() as tmp:
        objects = [os.path.join(tmp, s + ".o") for s in SOURCES]

        def compile_one(pair):
            cmd = [hipcc] + HIPCC_FLAGS + ["-c", os.path.join(CSRC, pair[0]), "-o", pair[1]]
            if verbose:
                print(" ".join(cmd), flush=True)
            subprocess.check_call(cmd)

        with ThreadPoolExecutor(max_workers=min(8, os.cpu_count() or 1)) as pool:
            list(pool.map(compile_one, zip(SOURCES, objects)))
        subprocess.check_call([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objects + ["-o", LIB])
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
