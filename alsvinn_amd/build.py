"""Build libalsvinn_hip.so (the hip platform) for gfx950 with hipcc.

Every HIP source is compiled with -ffp-contract=off (the FP64 stage must
keep the reference's rounding: no FMA contraction), without fast-math, and
with packed FP32 disabled.  Objects go to alsvinn_amd/_build/, the library
next to this file so that it travels with the source tree.
"""
import concurrent.futures
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libalsvinn_hip.so")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

SOURCES = [
    "avh_capi.hip",
    "avh_uq.hip",
    "avh_mlp.hip",
    "avh_volume.hip",
    "avh_stage_burgers.hip",
    "avh_stage_euler1.hip",
    "avh_stage_euler2.hip",
    "avh_stage_euler3.hip",
    "avh_stage_euler3_none.hip",
    "avh_stage_euler3_weno2.hip",
    "avh_stage_euler3_eno2.hip",
    "avh_stage_euler3_eno3.hip",
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
CFLAGS = [
    "--offload-arch=" + ARCH,
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", INCLUDE,
    "-Wall",
    "-Wno-unused-function",
]


def _compile(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + CFLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, " ".join(cmd), r.stderr))
    return obj


def build(verbose=False):
    """Compile every source and link the shared library.  Always rebuilds."""
    os.makedirs(BUILD, exist_ok=True)
    jobs = min(len(SOURCES), max(1, min(8, os.cpu_count() or 1)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(_compile, reversed(SOURCES)))  # the longest first
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=" + ARCH, "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (" ".join(cmd), r.stderr))
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
