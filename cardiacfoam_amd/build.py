"""Builds libcardiacgpu.so (HIP, gfx950) in-tree with hipcc.

Each .hip source compiles to an object in parallel, then one shared library is
linked next to this file.  Run as ``python -m cardiacfoam_amd.build``.
"""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import tempfile

from .listing import masked_reads

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libcardiacgpu.so")
SOURCES = ["model_fp64_ode.hip", "model_fp32_ode.hip", "model_fp64.hip", "model_fp32.hip",
           "tissue_implicit.hip", "ldu_solver.hip", "adjoint.hip", "ecg.hip",
           "general_mesh.hip", "capi.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
    # packed fp32 instructions are kept out of every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]

# Single-precision model kernels: reciprocal-based division, hardware exp2/log2 and
# fp32 denormals flushed to zero (fp64 keeps IEEE denormals; no finite-math assumption,
# so inf/NaN propagate as in IEEE arithmetic).
FAST_F32 = [
    "-fno-hip-fp32-correctly-rounded-divide-sqrt", "-fno-math-errno", "-freciprocal-math",
    "-fapprox-func", "-fno-signed-zeros", "-fgpu-flush-denormals-to-zero",
]
# FP64 Rush-Larsen kernels: instruction selection ordered for register pressure.  With the
# default source order ORd's tissue kernel spills 167 registers per lane, with this one 39.
LOW_PRESSURE = ["-mllvm", "-pre-RA-sched=list-burr"]
# With many scalar spills this compiler can put a vector register's copy ahead of a restored
# execution mask (listing.py).  Either of these leaves no such copy in the FP64 model kernels:
# scalar registers allocated without live-range splitting, or loop-invariant values not moved
# out of loops (fewer live registers).  The adaptive unit takes the second: under the first
# one state of Gaur's RKF45 cell kernel is wrong, for a cause that the listing does not show.
SAFE_SPILLS = ["-mllvm", "-sgpr-regalloc=basic"]
NO_HOISTS = ["-mllvm", "-disable-machine-licm"]
EXTRA = {"model_fp64.hip": LOW_PRESSURE + SAFE_SPILLS, "model_fp64_ode.hip": NO_HOISTS,
         "model_fp32.hip": FAST_F32, "model_fp32_ode.hip": FAST_F32}


def _compile(src):
    obj = os.path.join(BUILD, src.replace(".hip", ".o"))
    # in a folder of its own, with the intermediate files: the device listing among them is
    # looked over before it goes
    tmp = tempfile.mkdtemp(dir=BUILD)
    try:
        cmd = [HIPCC, *FLAGS, *EXTRA.get(src, []), "--save-temps=obj", "-c",
               os.path.join(CSRC, src), "-o", os.path.join(tmp, os.path.basename(obj))]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("hipcc failed for %s:\n%s\n%s" % (src, " ".join(cmd), r.stderr))
        listings = [f for f in os.listdir(tmp) if f.endswith(".s") and "amdgcn" in f]
        if not listings:
            raise RuntimeError("no device listing of %s" % src)
        for f in listings:
            bad = masked_reads(os.path.join(tmp, f))
            if bad:
                raise RuntimeError("%s: registers copied under the wrong lanes in %s" %
                                   (src, ", ".join("%s %s" % (k, v[:3]) for k, v in bad.items())))
        os.replace(os.path.join(tmp, os.path.basename(obj)), obj)
    finally:
        shutil.rmtree(tmp, ignore_errors=True)
    return obj


def build(verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s" % r.stderr)
    os.replace(tmp, LIB)
    if verbose:
        print("built", LIB)
    return LIB


if __name__ == "__main__":
    build()
    sys.exit(0)
