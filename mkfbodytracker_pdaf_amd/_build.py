"""In-tree build of the gfx950 shared library ``libmkfbt.so``.

The library is compiled with hipcc for gfx950 only.  Packed FP32 VALU ops are
disabled (``-packed-fp32-ops``) for all device code.
"""
from __future__ import annotations

import os
import subprocess

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.environ.get("MKFBT_LIB") or os.path.join(HERE, "libmkfbt.so")
SOURCES = ["pf_capi.hip", "pf_step_rec.hip", "pf_step_rows.hip", "pf_model.cpp", "pf_io.cpp", "pf_host.cpp", "pf2d.hip", "pf_batch.hip", "pf_adjoint.hip", "pf_tracker.hip", "pf_noalloc.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         # the joint loop of the widest kernels (8 joints of d = 16, two particles per
         # lane) exceeds the default size for full unrolling, and the state of a loop
         # that is not unrolled lives in scratch memory
         "-mllvm", "-pragma-unroll-threshold=65536",
         "-Wall", "-Wno-unused-function", "-Wno-unused-command-line-argument"]


def sources():
    return [os.path.join(CSRC, s) for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]


def build(verbose: bool = False, jobs: int = 0) -> str:
    """Compile every source under csrc/ into libmkfbt.so (always rebuilds):
    one hipcc per source in parallel, then one link."""
    import tempfile
    from concurrent.futures import ThreadPoolExecutor

    tmp = LIB + ".tmp"
    inc = ["-I", os.path.join(HERE, "..", "include")]
    cflags = [f for f in FLAGS if f != "-shared"]
    with tempfile.TemporaryDirectory(prefix="mkfbt_build_") as objdir:
        srcs = sources()
        objs = [os.path.join(objdir, os.path.basename(s) + ".o") for s in srcs]

        def compile_one(so):
            src, obj = so
            return subprocess.run([HIPCC, *cflags, *inc, "-c", src, "-o", obj], capture_output=True, text=True)

        n = jobs or min(len(srcs), os.cpu_count() or 1, 16)
        with ThreadPoolExecutor(max_workers=max(1, n)) as ex:
            results = list(ex.map(compile_one, zip(srcs, objs)))
        for src, res in zip(srcs, results):
            if res.returncode != 0:
                raise RuntimeError(f"hipcc failed on {os.path.basename(src)}:\n" + res.stderr[-8000:])
            if verbose and res.stderr:
                print(res.stderr)
        res = subprocess.run([HIPCC, *FLAGS, *objs, "-o", tmp], capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError("link failed:\n" + res.stderr[-8000:])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
