"""Builds chadslab_amd/libchadq.so from csrc/*.hip with hipcc for gfx950 (cross-compiles without a GPU).

Run as `python -m chadslab_amd.build` or through __graft_entry__.build().  The library is kept in-tree,
next to this file, with the torch extension of ops.py beside it (`--lib-only`: without); nothing is installed.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OBJ = PKG / "csrc" / "_obj"
LIB = PKG / "libchadq.so"
HOST = PKG / "_host_call.so"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
# -packed-fp32-ops: keep the compiler from forming packed fp32 arithmetic (v_pk_*_f32)
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc", "-Wall", "-Wno-unused-function",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # the first 16 dwords of a kernel's arguments arrive in scalar registers with the wave instead of being fetched
    # by its first instructions: these kernels last 3-10 us and every one of them starts by waiting for that fetch
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
]


def _run(cmd):
    p = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass does not know the packed-fp32 feature and says so on every file: drop that line
    err = "\n".join(l for l in p.stderr.splitlines() if "packed-fp32-ops" not in l)
    if p.returncode != 0:
        raise RuntimeError("command failed: %s\n%s\n%s" % (" ".join(map(str, cmd)), p.stdout, err))
    if err.strip():
        sys.stderr.write(err + "\n")


def build_host(verbose: bool = True) -> Path:
    """csrc/host_call.cpp -> _host_call.so: the plain calls of ops.py in C++ (host code only, against torch's own headers)."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    inc = [sysconfig.get_paths()["include"], *cpp_extension.include_paths(), "/opt/rocm/include"]
    lib = str(Path(torch.__file__).resolve().parent / "lib")
    tmp = HOST.with_suffix(".so.tmp")
    # NDEBUG: without it pybind11's headers put a thread-local counter into the module.  A module with thread-local storage that is opened
    # late and whose storage nobody touches leaves every thread's table behind the loader's count, and from then on each look at
    # thread-local storage in all other libraries (torch's current device and stream, its allocator) takes the loader's slow way:
    # torch.empty 1.36 -> 1.65 us, a product through ctypes 6.6 -> 7.6
    _run([os.environ.get("CXX", "g++"), "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), *("-isystem%s" % i for i in inc),
          str(CSRC / "host_call.cpp"), "-o", str(tmp), "-L" + lib, "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"])
    os.replace(tmp, HOST)
    if verbose:
        print("built %s" % HOST)
    return HOST


def build(verbose: bool = True, save_temps: bool = False, host: bool = True) -> Path:
    """The library, its measurement builds and (host) the torch extension.  The library needs hipcc only and is linked whether or not the
    extension, which needs torch's and Python's headers and g++, can be built; what went wrong there is raised at the end."""
    srcs = sorted(CSRC.glob("*.hip"))
    if not srcs:
        raise RuntimeError("no HIP sources under %s" % CSRC)
    OBJ.mkdir(exist_ok=True)
    objs = [OBJ / (s.stem + ".o") for s in srcs]

    def one(pair):
        s, o = pair
        cmd = [HIPCC, *FLAGS, "-c", str(s), "-o", str(o)]
        if save_temps:
            cmd += ["-save-temps=obj"]
        _run(cmd)
        return o

    with ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        extension = ex.submit(build_host, verbose) if host else None
        list(ex.map(one, zip(srcs, objs)))
    tmp = LIB.with_suffix(".so.tmp")
    _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, LIB)
    if verbose:
        print("built %s (%d sources)" % (LIB, len(srcs)))
    build_ablations(verbose)  # always together: the measurement builds share every other object and the whole C ABI
    if extension is not None:
        extension.result()
    return LIB


# Measurement builds (bench.py --extras moe_ablation / gemm_ablation): the same library with a part of one kernel's loop
# compiled out, so that the part's share of the time can be measured on its own.  Their results are wrong by
# construction; nothing but the bench loads them.  name -> (source file, macro definition)
ABLATIONS = {"stream": ("gemm_expert_i4g32.hip", "-DCHADQ_EXPERT_ABLATE=1"),   # expert GEMM: memory traffic without arithmetic
             "arith": ("gemm_expert_i4g32.hip", "-DCHADQ_EXPERT_ABLATE=2"),    # expert GEMM: arithmetic without weight loads
             "nodequant": ("gemm_tile_q.hip", "-DCHADQ_GEMM_ABLATE=1")}        # prefill GEMM: no dequantisation


def ablation_path(name: str) -> Path:
    return PKG / ("libchadq_ablate_%s.so" % name)


def build_ablations(verbose: bool = True) -> None:
    """Only the one source file of each ablation is recompiled; the other objects are those of the library."""
    def one(item):
        name, (fname, define) = item
        src = CSRC / fname
        obj = OBJ / ("ablate_%s.o" % name)
        _run([HIPCC, *FLAGS, define, "-c", str(src), "-o", str(obj)])
        return name, src, obj

    with ThreadPoolExecutor(max_workers=len(ABLATIONS)) as ex:
        done = list(ex.map(one, ABLATIONS.items()))
    for name, src, obj in done:
        others = [o for o in sorted(OBJ.glob("*.o")) if o.stem != src.stem and not o.stem.startswith("ablate_") and
                  (CSRC / (o.stem + ".hip")).exists()]
        tmp = ablation_path(name).with_suffix(".so.tmp")
        _run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, others), str(obj)])
        os.replace(tmp, ablation_path(name))
        if verbose:
            print("built %s" % ablation_path(name))


if __name__ == "__main__":
    build(save_temps="--save-temps" in sys.argv, host="--lib-only" not in sys.argv)
