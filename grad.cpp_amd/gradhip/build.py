"""Builds libgradhip.so (HIP kernels + C ABI) for gfx950 with hipcc, in-tree."""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CSRC = os.path.join(PKG, "csrc")
LIB_DIR = os.path.join(PKG, "lib")
LIB = os.path.join(LIB_DIR, "libgradhip.so")

# -packed-fp32-ops is switched off on purpose: some packed fp32 forms have given
# wrong results on this hardware pool.  No fast-math: GELU/SiLU/softmax/RoPE use
# the precise expf/tanhf.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-fast-math", "-Wall", "-Wno-unused-function", *os.environ.get("GRADHIP_EXTRA_FLAGS", "").split(),
]
SOURCES = ["engine.hip", "persist.hip", "xcd.hip", "resident.hip", "rows.hip", "pairs.hip", "checkpoint.cpp", "tokenizer.cpp"]
OBJ_DIR = os.path.join(PKG, "build")


BIN_DIR = os.path.join(PKG, "bin")
CLI = os.path.join(BIN_DIR, "gradhip-generate")
INCLUDE = os.path.join(os.path.dirname(PKG), "include")


def build(verbose: bool = True) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(OBJ_DIR, exist_ok=True)

    def compile_one(src: str) -> str:
        obj = os.path.join(OBJ_DIR, src + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
        return obj

    # the translation units do not share device code: compile them side by side
    with ThreadPoolExecutor(len(SOURCES)) as pool:
        objs = list(pool.map(compile_one, SOURCES))
    subprocess.check_call([hipcc, "--offload-arch=gfx950", "-shared", "-o", LIB, *objs])
    # the command-line caller: plain C++ over the header-only adapter
    os.makedirs(BIN_DIR, exist_ok=True)
    for src, exe in (("generate.cpp", CLI), ("chat.cpp", os.path.join(BIN_DIR, "gradhip-chat")),
                     ("bench.cpp", os.path.join(BIN_DIR, "gradhip-bench")),
                     ("eval.cpp", os.path.join(BIN_DIR, "gradhip-eval"))):
        cmd = ["g++", "-std=c++20", "-O2", "-Wall", "-Wextra", "-I", INCLUDE, os.path.join(PKG, "cli", src),
               "-o", exe, "-L", LIB_DIR, "-lgradhip", "-Wl,-rpath,$ORIGIN/../lib"]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
