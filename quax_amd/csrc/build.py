"""Builds libquax_hip.so for gfx950.

Steps: generate the per-class kernel sources (gen_eri.py) into csrc/_gen,
compile every translation unit with hipcc in parallel, link the shared
library into quax_amd/lib/.  Objects are cached under csrc/_build keyed by a
hash of (source, headers, flags); ``force=True`` recompiles everything.

Usage: python -m quax_amd.csrc.build [--force] [--jobs N] [--lmax L] [--no-fp32] [--budget N] [--out PATH]
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import hashlib
import os
import re
import shutil
import subprocess
import sys
import tempfile
import time

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
GEN = os.path.join(HERE, "_gen")
OBJ = os.path.join(HERE, "_build")
LIBDIR = os.path.join(PKG, "lib")
LIB = os.path.join(LIBDIR, "libquax_hip.so")
ROOT = os.path.dirname(PKG)

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
ARCH = "gfx950"
FLAGS = ["-std=c++17", "-O3", f"--offload-arch={ARCH}", "-fPIC", "-munsafe-fp-atomics",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-variable", "-Wno-unused-but-set-variable",
         f"-I{os.path.join(ROOT, 'include')}", f"-I{HERE}"]

RUNTIME_SOURCES = ["qx_runtime.hip", "qx_kernels.hip", "qx_jk.hip", "qx_gemm.hip", "qx_scf.hip"]
HEADERS = ["qx_device.h", "qx_pairm.h", "qx_jk.h", "qx_grad.h", "qx_rys.h", "qx_oei.h", "qx_runtime.h"]
# what each header of the generated sources stands for, besides qx_device.h
INCLUDES = {"qx_device.h": [], "qx_pairm.h": ["qx_pairm.h"], "qx_jk.h": ["qx_jk.h"], "qx_grad.h": ["qx_grad.h", "qx_jk.h"],
            "qx_rys.h": ["qx_rys.h", "qx_grad.h", "qx_jk.h", "qx_pairm.h"],
            "qx_oei.h": ["qx_oei.h", "qx_runtime.h", "qx_pairm.h", "qx_jk.h"]}


def _hash(paths, extra):
    h = hashlib.sha256()
    for p in paths:
        with open(p, "rb") as fh:
            h.update(fh.read())
    h.update(" ".join(extra).encode())
    return h.hexdigest()[:20]


def _flags(src):
    """Compiler flags of one translation unit: the runtime sources also see
    the generated class tables (qx_classes.inc in GEN)."""
    return _opt_flags(src) if src.startswith(GEN) else FLAGS + [f"-I{GEN}"]


def _opt_flags(src):
    """Dual-number kernels (second derivatives), the ones that spill, build at
    -O2: at -O3 the gfx950 compiler returned a wrong value for one element of
    an inlined (dd|ps) tangent kernel that was right at -O2, built with g++ on
    the host and evaluated in Python."""
    name = os.path.basename(src)
    if name.startswith("jengv_") or name.split("_")[-1].startswith("v"):
        return [f if f != "-O3" else "-O2" for f in FLAGS]
    return FLAGS


def _compile(src, force):
    if src.startswith(GEN):
        # generated class kernels depend on the header they include and on
        # qx_device.h (the class tables in qx_classes.inc are compiled into
        # qx_runtime.hip alone)
        with open(src) as fh:
            first = re.match(r'#include "\.\./(\w+\.h)"', fh.readline())
        heads = {"qx_device.h"} | set(INCLUDES[first.group(1)])
        deps = [src] + sorted(os.path.join(HERE, h) for h in heads)
    else:
        deps = [src] + [os.path.join(HERE, h) for h in HEADERS] + [os.path.join(ROOT, "include", "quax_amd.h"),
                                                                   os.path.join(GEN, "qx_classes.inc")]
    flags = _flags(src)
    key = _hash([d for d in deps if os.path.exists(d)], flags)
    obj = os.path.join(OBJ, os.path.basename(src) + "." + key + ".o")
    if os.path.exists(obj) and not force:
        return obj, 0.0, True
    t0 = time.time()
    cmd = [HIPCC] + flags + ["-c", src, "-o", obj + ".tmp"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-4000:]}")
    os.replace(obj + ".tmp", obj)
    return obj, time.time() - t0, False


H5_PREFIX = os.environ.get("QX_HDF5_PREFIX", "/opt/conda")
H5_LIB = os.path.join(LIBDIR, "libquax_h5.so")


def build_h5(verbose=True):
    """libquax_h5.so (HDF5 files of the disk mode): host C on the HDF5 C
    library under QX_HDF5_PREFIX (default /opt/conda); skipped with a message
    when that library is absent."""
    inc, lib = os.path.join(H5_PREFIX, "include"), os.path.join(H5_PREFIX, "lib")
    if not (os.path.exists(os.path.join(inc, "hdf5.h")) and os.path.exists(os.path.join(lib, "libhdf5.so"))):
        if verbose:
            print(f"  HDF5 not found under {H5_PREFIX}: libquax_h5.so (disk mode) not built", flush=True)
        return None
    os.makedirs(LIBDIR, exist_ok=True)
    cmd = ["gcc", "-O2", "-shared", "-fPIC", "-Wall", f"-I{os.path.join(ROOT, 'include')}", f"-I{inc}",
           os.path.join(HERE, "qx_h5.c"), f"-L{lib}", "-lhdf5", f"-Wl,-rpath,{lib}", "-o", H5_LIB + ".tmp"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"gcc failed for qx_h5.c:\n{r.stderr[-4000:]}")
    os.replace(H5_LIB + ".tmp", H5_LIB)
    if verbose:
        print(f"built {H5_LIB}", flush=True)
    return H5_LIB


# Scratch per lane allowed to the generated kernels, which run on up to four
# streams: a side stream's hardware queue that has to
# grow its scratch past ~8 KB per lane, once the process holds scratch on its
# other queues, has been refused by the HSA runtime (the queue aborts with
# HSA_STATUS_ERROR_OUT_OF_RESOURCES).  The caller's stream is no safer: nothing
# a context runs before grows its scratch.
STREAMING_SCRATCH_MAX = 6144
LLVM_BIN = os.path.join(ROCM, "llvm", "bin")
# Scratch per lane of the kernels that hold their lists as one kernel argument,
# as built without a copy of that argument in scratch.  A dual-number J kernel
# with such a copy (304 bytes more) returned wrong potentials.
ARGUMENT_SCRATCH = {"jk_small": 0, "grad_small": 232, "jeng_0": 0, "jeng_1": 0, "jeng_2": 0, "jeng_3": 0, "jeng_4": 448,
                    "jengv_0": 0, "jengv_1": 0, "jengv_2": 192, "jengv_3": 1432, "jengv_4": 3192}


def kernel_scratch(obj: str, tmp: str) -> list:
    """(kernel name, scratch bytes per lane) of the gfx950 code object in a
    compiled object file (its .hip_fatbin offload bundle)."""
    fb, co = os.path.join(tmp, "fb.bin"), os.path.join(tmp, "k.co")
    subprocess.run([os.path.join(LLVM_BIN, "llvm-objcopy"), f"--dump-section=.hip_fatbin={fb}", obj, os.devnull],
                   check=True, capture_output=True)
    subprocess.run([os.path.join(LLVM_BIN, "clang-offload-bundler"), "--unbundle", "--type=o", f"--input={fb}",
                    f"--targets=hipv4-amdgcn-amd-amdhsa--{ARCH}", f"--output={co}"], check=True, capture_output=True)
    notes = subprocess.run([os.path.join(LLVM_BIN, "llvm-readelf"), "--notes", co], check=True,
                           capture_output=True, text=True).stdout
    names = re.findall(r"\.name:\s+(\S+)", notes)
    sizes = [int(x) for x in re.findall(r"\.private_segment_fixed_size:\s+(\d+)", notes)]
    return list(zip(names, sizes))


def check_streaming_scratch(objs, verbose=True):
    """Fails the build when a generated kernel needs more than
    STREAMING_SCRATCH_MAX bytes of scratch per lane, or one of ARGUMENT_SCRATCH
    more than its bytes there."""
    if not os.path.exists(os.path.join(LLVM_BIN, "clang-offload-bundler")):
        print("scratch check skipped: no clang-offload-bundler", flush=True)
        return
    streaming = [o for o in objs if not os.path.basename(o).startswith("qx_")]
    worst, copies = ("", 0), []
    with tempfile.TemporaryDirectory() as tmp:
        for o in streaming:
            for name, size in kernel_scratch(o, tmp):
                if size > worst[1]:
                    worst = (name, size)
                if size > ARGUMENT_SCRATCH.get(os.path.basename(o).split(".hip.")[0], size):
                    copies.append((name, size))
    if worst[1] > STREAMING_SCRATCH_MAX:
        raise RuntimeError(f"streaming kernel {worst[0]} needs {worst[1]} B of scratch per lane "
                           f"(at most {STREAMING_SCRATCH_MAX} allowed on side streams)")
    if copies:
        raise RuntimeError(f"kernels with more scratch than without a copy of their arguments: {copies}")
    if verbose:
        print(f"streaming kernels: at most {worst[1]} B of scratch per lane ({worst[0]})", flush=True)


def build(force=False, jobs=None, lmax=2, fp32=True, verbose=True, budget=None, out=None, waves=None,
          csplit=None):
    """budget / waves: one derivative node budget / waves-per-SIMD target for
    every class instead of the tuned per-class table (tuning builds); out:
    library path."""
    lib = out or LIB
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(os.path.dirname(os.path.abspath(lib)), exist_ok=True)
    gen_args = [sys.executable, os.path.join(HERE, "gen_eri.py"), GEN, str(lmax)] + ([] if fp32 else ["--no-fp32"])
    env = dict(os.environ)
    env.pop("QX_DERIV_NODES", None)
    env.pop("QX_GRAD_WAVES", None)
    env.pop("QX_CSPLIT", None)
    if csplit:
        env["QX_CSPLIT"] = str(int(csplit))
    if budget:
        env["QX_DERIV_NODES"] = str(int(budget))
    if waves:
        env["QX_GRAD_WAVES"] = str(int(waves))
    if os.path.isdir(GEN):
        shutil.rmtree(GEN)
    subprocess.run(gen_args, check=True, capture_output=True, env=env)
    gen_srcs = sorted(os.path.join(GEN, f) for f in os.listdir(GEN) if f.endswith(".hip"))
    # biggest first so the long poles start early
    gen_srcs.sort(key=lambda p: -os.path.getsize(p))
    srcs = [os.path.join(HERE, s) for s in RUNTIME_SOURCES] + gen_srcs
    jobs = jobs or min(16, os.cpu_count() or 4)
    t0 = time.time()
    objs = []
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        futs = {ex.submit(_compile, s, force): s for s in srcs}
        for f in cf.as_completed(futs):
            obj, dt, cached = f.result()
            objs.append(obj)
            if verbose and not cached:
                print(f"  compiled {os.path.basename(futs[f])} in {dt:.1f} s", flush=True)
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", lib + ".tmp"] + sorted(objs)
    subprocess.run(cmd, check=True)
    check_streaming_scratch(objs, verbose)
    os.replace(lib + ".tmp", lib)
    if verbose:
        print(f"built {lib} ({len(objs)} objects, {time.time() - t0:.1f} s)", flush=True)
    if out is None:
        build_h5(verbose)
    return lib


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("--lmax", type=int, default=2)
    ap.add_argument("--no-fp32", action="store_true", help="skip the FP32 (mixed-precision) kernels")
    ap.add_argument("--budget", type=int, default=None,
                    help="one derivative node budget for all classes (tuning builds)")
    ap.add_argument("--waves", type=int, default=None,
                    help="one waves-per-SIMD target for all adjoint kernels (tuning builds)")
    ap.add_argument("--csplit", type=int, default=None,
                    help="c-component ranges per (a, b) derivative part for every class (tuning builds)")
    ap.add_argument("--out", default=None, help="library path (default quax_amd/lib/libquax_hip.so)")
    a = ap.parse_args()
    build(force=a.force, jobs=a.jobs, lmax=a.lmax, fp32=not a.no_fp32, budget=a.budget, out=a.out, waves=a.waves,
          csplit=a.csplit)
