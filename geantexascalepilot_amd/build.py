"""Build libgxt.so (HIP for gfx950) in-tree.

hipcc compiles the device code for gfx950 only.  FP contraction is off so the
FP64 arithmetic is rounded operation by operation as written, and packed FP32
instructions are disabled.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libgxt.so")
SOURCES = ["gxt_kernels.hip", "gxt_engine.cpp", "gxt_data.cpp", "gxt_events.cpp", "gxt_field.cpp", "gxt_nav.cpp"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wall", "-Wno-unused-parameter",
         "-Wno-unused-function"]


# The step loop is compiled once per precision and transport mode, each with
# its waves per workgroup (a quarter of them on each SIMD).  Without the
# machine-level hoisting of loop invariants, which moves the samplers'
# constants out of the loop over tasks into registers held for good: 225 to 180
# VGPRs for the plain FP64 loop.
LOOP_WAVES = {("double", 0): 12, ("double", 1): 12, ("double", 2): 8, ("double", 3): 8, ("double", 4): 8,
              ("float", 0): 12, ("float", 1): 12, ("float", 2): 12, ("float", 3): 8, ("float", 4): 12}
# (object, source, extra flags)
UNITS = [(os.path.splitext(f)[0], f, []) for f in SOURCES] + [
    ("gxt_loop_%s_%d" % k, "gxt_loop.hip",
     ["-DGXT_LOOP_R=" + k[0], "-DGXT_LOOP_MODE=%d" % k[1], "-DGXT_LOOP_WAVES=%d" % w,
      "-mllvm", "-disable-machine-licm"]) for k, w in sorted(LOOP_WAVES.items())]


def _compile(unit, build_dir, verbose):
    name, src, defs = unit
    obj = os.path.join(build_dir, name + ".o")
    cmd = [HIPCC] + (["-x", "hip"] if src.endswith(".cpp") else []) + FLAGS + defs + \
        ["-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd))
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed on %s:\n%s" % (src, r.stdout + r.stderr))
    return obj


def build(verbose=False):
    build_dir = os.path.join(HERE, "_build")
    os.makedirs(build_dir, exist_ok=True)
    with ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as ex:
        objs = list(ex.map(lambda u: _compile(u, build_dir, verbose), UNITS))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("link of libgxt.so failed")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
