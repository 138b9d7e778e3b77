"""Builds libodmkv.so (the HIP kernels and their C ABI) for gfx950 with hipcc, and
libodmkv_bench.so: the same object files plus the measurement entry points of csrc/bench_hooks.hip
(include/odmkv_bench.h), which the product library does not export; and kvquant/_native.so, the decode
step's host path over torch tensors.

    python odm-kv_amd/build.py [--force]

hipcc cross-compiles without a GPU.  Flags that matter:
  -ffp-contract=off   nothing is fused unless the source says fma: the allocator's cost and the
                      quantiser's rotation are bit-exact contracts with their CPU statements;
  packed-fp32-ops off the compiler must not form packed fp32 instructions.
Both libraries are linked with csrc/exports.map: only the C entry points (odmkv_*) are dynamic symbols.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libodmkv.so")
BENCH_LIB = os.path.join(LIBDIR, "libodmkv_bench.so")
SOURCES = ["error.hip", "score.hip", "window.hip", "allocate.hip", "pack.hip", "rows.hip", "decode.hip", "flush.hip", "codebook.hip",
           "levels.hip", "query_stats.hip", "store_edit.hip", "worklist.cpp"]
BENCH_SOURCES = ["bench_hooks.hip"]
NATIVE = os.path.join(HERE, "kvquant", "_native.so")          # the CPython extension of csrc/torch_step.cpp (host code only)
FLAGS = [
    "-O3", "--offload-arch=gfx950", "-fPIC", "-std=c++17", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]


def _newest(paths):
    return max(os.path.getmtime(p) for p in paths)


def _build_native(verbose: bool) -> None:
    import importlib.util
    import sysconfig
    torch_dir = os.path.dirname(importlib.util.find_spec("torch").origin)
    cmd = ["g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-I" + os.path.join(torch_dir, "include"),
           "-I" + os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"), "-I" + sysconfig.get_paths()["include"],
           os.path.join(CSRC, "torch_step.cpp"), "-o", NATIVE, "-L" + os.path.join(torch_dir, "lib"), "-lc10", "-ltorch",
           "-ltorch_cpu", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on torch_step.cpp:\n{r.stdout}\n{r.stderr}")


def build(force: bool = False, verbose: bool = True) -> str:
    srcs = [os.path.join(CSRC, s) for s in SOURCES + BENCH_SOURCES]
    deps = srcs + [os.path.join(CSRC, "torch_step.cpp")] + [os.path.join(CSRC, h) for h in ("common.h", "quant.h", "decode.h", "exports.map")] + [
        os.path.join(HERE, "..", "include", "odmkv.h"), os.path.join(HERE, "..", "include", "odmkv_bench.h"), __file__]
    if (not force and os.path.exists(LIB) and os.path.exists(BENCH_LIB) and os.path.exists(NATIVE)
            and min(map(os.path.getmtime, (LIB, BENCH_LIB, NATIVE))) >= _newest(deps)):
        return LIB
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)

    def compile_one(src):
        obj = os.path.join(objdir, os.path.basename(src) + ".o")
        cmd = ["hipcc", *FLAGS, "-c", src, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
        warn = [ln for ln in r.stderr.splitlines() if "packed-fp32-ops" not in ln and ln.strip()]
        if warn and verbose:
            print("\n".join(warn))
        return obj

    with ThreadPoolExecutor(max_workers=8) as ex:
        native = ex.submit(_build_native, verbose)
        objs = list(ex.map(compile_one, srcs))
        native.result()
    product = objs[:len(SOURCES)]
    for lib, parts in ((LIB, product), (BENCH_LIB, objs)):
        cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", f"-Wl,--version-script={os.path.join(CSRC, 'exports.map')}",
               "-o", lib, *parts]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    return LIB


if __name__ == "__main__":
    print(build(force="--force" in sys.argv))
