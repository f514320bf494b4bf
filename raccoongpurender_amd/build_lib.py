"""Compile the gfx950 HIP library (libraccoongpu.so) in-tree with hipcc.

Used by __graft_entry__.build(); also runnable as `python -m raccoongpurender_amd.build_lib`.
"""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libraccoongpu.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

SOURCES = ["capi.cpp", "bvh_build.cpp", "bvh_gpu.hip", "envmap_build.cpp", "scene_pack.hip", "traverse.hip", "util.hip", "wavefront.hip", "wavefront_capi.cpp", "guide.hip"]

# -ffp-contract=off keeps every float expression unfused so results match the CPU
# oracle bit for bit; packed fp32 instructions are disabled for correctness.
COMMON = [
    "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]
DEVICE = [
    "--offload-arch=gfx950",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# Correctly rounded fp32 division and square root wherever results are compared with the
# oracle bit for bit; the network kernels (guide.hip) are checked to a tolerance instead.
EXACT = ["-fhip-fp32-correctly-rounded-divide-sqrt"]
TOLERANT = {"guide.hip"}


def build(verbose: bool = False, jobs: int = 8) -> str:
    objdir = os.path.join(HERE, "_build")
    os.makedirs(objdir, exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES:
        path = os.path.join(CSRC, src)
        obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
        objs.append(obj)
        flags = [*COMMON, *DEVICE, *([] if src in TOLERANT else EXACT)]
        if src.endswith(".hip"):
            cmd = [HIPCC, "-x", "hip", *flags, "-c", path, "-o", obj]
        else:
            cmd = [HIPCC, *flags, "-c", path, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        if len([p for p in procs if p[1].poll() is None]) >= jobs:
            procs[0][1].wait()
    failed = []
    for src, p in procs:
        out, _ = p.communicate()
        text = out.decode(errors="replace")
        if p.returncode != 0:
            failed.append((src, text))
        elif verbose and text.strip():
            print(text)
    if failed:
        for src, text in failed:
            sys.stderr.write(f"--- {src}\n{text}\n")
        raise RuntimeError("HIP library build failed: " + ", ".join(s for s, _ in failed))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs, "-lpthread"]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
