"""Builds libdqmc_hip.so (the C-ABI library) in-tree with hipcc for gfx950.

Every .hip source under dqmc_amd/csrc is compiled to an object in parallel and
linked into dqmc_amd/_lib/libdqmc_hip.so. Run as `python -m dqmc_amd.build`.
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
SRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_lib")
LIB = os.path.join(OUT_DIR, "libdqmc_hip.so")
ARCH = os.environ.get("DQMC_OFFLOAD_ARCH", "gfx950")

FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=" + ARCH,
    # packed FP32 instructions stay disabled in all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]

# The windowed local-update kernel holds many phases in one loop nest: hoisting their constants
# and lane addresses out of it spills 27 registers into the loop that decides proposals
# (reloads of some 800 cycles each on its serial chain); without the hoisting the instance with
# LDS-resident columns spills none and the other one 4 (20 bytes per lane).
FILE_FLAGS = {"k_local.hip": ["-mllvm", "-disable-machine-licm"]}


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found")


def _compile(src, obj):
    cmd = [hipcc()] + FLAGS + FILE_FLAGS.get(os.path.basename(src), []) + ["-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("compile failed: %s\n%s\n%s" % (" ".join(cmd), r.stdout, r.stderr))
    return obj


def build(verbose=False):
    os.makedirs(OUT_DIR, exist_ok=True)
    objdir = os.path.join(OUT_DIR, "obj")
    os.makedirs(objdir, exist_ok=True)
    srcs = sorted(f for f in os.listdir(SRC) if f.endswith(".hip"))
    jobs = []
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        for f in srcs:
            obj = os.path.join(objdir, f[:-4] + ".o")
            jobs.append(ex.submit(_compile, os.path.join(SRC, f), obj))
        objs = [j.result() for j in jobs]
    tmp = LIB + ".tmp"
    cmd = [hipcc(), "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed: %s\n%s" % (r.stdout, r.stderr))
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
