"""Builds libtalos_hip.so (the C-ABI library) from csrc/*.hip with hipcc for gfx950.

Each translation unit is compiled to an object in parallel, then the objects are linked into
talos-xii_amd/libtalos_hip.so next to this file (in-tree, so it travels with the repository).
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libtalos_hip.so")
ARCH = "gfx950"

HIP_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # no packed-fp32 (v_pk_*_f32) instructions anywhere in the device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result", "-Wno-unused-variable",
]


# Flags of single sources. acnet.hip: its one loop covers the whole kernel, and hoisting the f64 loss's
# constants out of it costs 60 registers over every phase (254 of 258 VGPR spills were theirs).
SOURCE_FLAGS = {"acnet.hip": ["-mllvm", "-disable-machine-licm"]}


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src):
    obj = os.path.join(BUILD, os.path.basename(src) + ".o")
    cmd = ["hipcc", *HIP_FLAGS, *SOURCE_FLAGS.get(os.path.basename(src), []), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    return obj, r.stderr


def build(verbose=False, jobs=None):
    """Compiles every csrc/*.hip and links libtalos_hip.so. Always rebuilds."""
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    jobs = jobs or min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with concurrent.futures.ThreadPoolExecutor(jobs) as ex:
        results = list(ex.map(_compile, srcs))
    objs = []
    for obj, err in results:
        objs.append(obj)
        if verbose and err.strip():
            print(err, file=sys.stderr)
    tmp = LIB + ".tmp"
    cmd = ["hipcc", f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    build_tape()
    return LIB


TAPE_SRC = os.path.join(HERE, "host", "tape.cpp")
TAPE_LIB = os.path.join(HERE, "libtalos_tape.so")


def build_tape():
    """Builds libtalos_tape.so, the host-side C++ tape (host/tape.cpp) over the C ABI."""
    tmp = TAPE_LIB + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", TAPE_SRC, "-o", tmp, f"-L{HERE}", "-ltalos_hip",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for {TAPE_SRC}:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, TAPE_LIB)
    return TAPE_LIB


if __name__ == "__main__":
    print(build(verbose=True))
