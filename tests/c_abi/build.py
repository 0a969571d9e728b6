"""Builds the C++ programs that the tests run: abi_check.out, the C ABI exercised from plain C++
(hipcc host compile, linked against the in-tree libbutterfly_hip.so and, as the checker,
oracle/liboracle.so), and reduce_check.out, host arithmetic of the reduce (no GPU)."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(os.path.dirname(HERE))
OUT = os.path.join(HERE, "abi_check.out")
REDUCE = os.path.join(HERE, "reduce_check.out")
HIPCC = ["hipcc", "-std=c++17", "--offload-arch=gfx950", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]


def build():
    build_reduce()
    cmd = HIPCC + ["-O2", os.path.join(HERE, "abi_check.cpp"),
           "-I", os.path.join(ROOT, "include"),
           "-L", os.path.join(ROOT, "butterfly_amd"), "-lbutterfly_hip",
           "-L", os.path.join(ROOT, "oracle"), "-loracle",
           "-Wl,-rpath,$ORIGIN/../../butterfly_amd", "-Wl,-rpath,$ORIGIN/../../oracle",
           "-o", OUT]
    print("+", " ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return OUT


def build_reduce():
    # (unoptimised: arithmetic whose result goes unused is done all the same)
    cmd = HIPCC + ["-O0", os.path.join(HERE, "reduce_check.cpp"), "-o", REDUCE]
    print("+", " ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    return REDUCE


if __name__ == "__main__":
    build()
    sys.exit(0)
