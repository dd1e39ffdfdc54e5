"""Build libpagedkv.so (the HIP kernels + C ABI) for gfx950 with hipcc.

Usage: python build_native.py [--jobs N]

Every `csrc/*.hip` file is compiled to an object under `_build/` and linked
into `lib/libpagedkv.so` next to this file; `csrc/bind.cpp` (the Python calls
into it) becomes `lib/_pkvbind.so` with the host compiler. hipcc cross-compiles, so this runs
on a machine without a GPU. Packed-FP32 instruction selection is switched off
for the device code (`-packed-fp32-ops`).
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libpagedkv.so")
BIND = os.path.join(LIBDIR, "_pkvbind.so")
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")
CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(HERE, "..", "include"),
]


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature;
    # keep every other diagnostic visible.
    err = "\n".join(
        ln for ln in res.stderr.splitlines()
        if "packed-fp32-ops" not in ln and "not a recognized feature" not in ln
    ).strip()
    if res.returncode != 0:
        raise RuntimeError(f"command failed ({res.returncode}): {' '.join(cmd)}\n{res.stderr}")
    if err:
        print(err, file=sys.stderr)


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip")
    )


def build(jobs: int = 4, verbose: bool = False) -> str:
    """Compile every kernel source and link lib/libpagedkv.so; returns its path."""
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(BUILD, os.path.basename(s)[:-4] + ".o") for s in srcs]

    def compile_one(pair):
        src, obj = pair
        cmd = [HIPCC, *CFLAGS, "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd))
        _run(cmd)
        return obj

    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        list(ex.map(compile_one, zip(srcs, objs)))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, LIB)
    build_bind()
    return LIB


def build_bind() -> None:
    """Compile lib/_pkvbind.so. Without a host compiler or Python's headers there
    is none, and the wrappers call the library through ctypes."""
    include = sysconfig.get_paths()["include"]
    if not shutil.which(CXX) or not os.path.exists(os.path.join(include, "Python.h")):
        print(f"no {CXX} or no Python.h in {include}: {BIND} is not built")
        if os.path.exists(BIND):
            os.remove(BIND)
        return
    tmp = BIND + ".tmp"
    _run([CXX, "-O2", "-fPIC", "-shared", "-std=c++17", "-Wall", "-I", include,
          os.path.join(CSRC, "bind.cpp"), "-o", tmp])
    os.replace(tmp, BIND)


def clean() -> None:
    shutil.rmtree(BUILD, ignore_errors=True)


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    ap.add_argument("--clean", action="store_true")
    ap.add_argument("-v", "--verbose", action="store_true")
    args = ap.parse_args()
    if args.clean:
        clean()
    print(build(args.jobs, args.verbose))
