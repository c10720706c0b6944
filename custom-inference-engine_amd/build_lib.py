"""Builds libcie_attn.so (the gfx950 attention library) in-tree.

    python custom-inference-engine_amd/build_lib.py              # the library
    python custom-inference-engine_amd/build_lib.py --timeline   # its timeline build

Every source is compiled for gfx950 with hipcc (objects under ``_build/``,
compiled in parallel) and linked into ``custom-inference-engine_amd/libcie_attn.so``,
which the Python layer loads with ctypes and calls through ``cie_host.so``. Packed-FP32 VALU instructions are
disabled for all device code.
"""

from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
INCLUDE = os.path.join(REPO, "include")
BUILD = os.path.join(PKG_DIR, "_build")
LIB_PATH = os.path.join(PKG_DIR, "libcie_attn.so")
HOST_PATH = os.path.join(PKG_DIR, "cie_host.so")  # CPython extension: the Python layer's calls into the library
TIMELINE_LIB_PATH = os.path.join(PKG_DIR, "libcie_attn_timeline.so")
# stand-alone microbenchmarks (benchmarks/<name>.hip -> _build/<name>), not part of the library
BENCH_TOOLS = ("vector_rates", "read_floor", "prefill_step")

SOURCES = ["capi.cpp", "paged_plan.cpp", "flash_fwd.hip", "paged_fwd.hip", "kv_append.hip", "rope.hip",
           "int8_gemm.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
COMMON = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # MFMA accumulators in VGPRs: the online-softmax rescale multiplies them on the VALU
    "-Xarch_device", "-mllvm=-amdgpu-mfma-vgpr-form=1",
    f"-I{INCLUDE}",
    f"-I{CSRC}",
]


def _run(cmd: list[str]) -> None:
    res = subprocess.run(cmd, capture_output=True, text=True)
    # hipcc's host pass does not know the packed-fp32 feature; that warning is noise
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"command failed ({res.returncode}): {' '.join(cmd)}\n{err}\n{res.stdout}")
    if err.strip():
        sys.stderr.write(err + "\n")


def _build_lib(out: str, objdir: str, defines: list[str]) -> None:
    os.makedirs(objdir, exist_ok=True)
    objs = []
    cmds = []
    for src in SOURCES:
        obj = os.path.join(objdir, os.path.splitext(src)[0] + ".o")
        lang = ["-x", "hip"] if src.endswith(".hip") else []
        cmds.append([HIPCC, *COMMON, *defines, *lang, "-c", os.path.join(CSRC, src), "-o", obj])
        objs.append(obj)
    with ThreadPoolExecutor(max_workers=min(len(cmds), os.cpu_count() or 1)) as ex:
        list(ex.map(_run, cmds))
    tmp = out + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, out)


def _build_host() -> None:
    """csrc/host.cpp against torch's C++ headers (host code only)."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths, library_paths

    inc = [f"-I{d}" for d in (INCLUDE, sysconfig.get_paths()["include"], "/opt/rocm/include")]
    inc += [f"-isystem{d}" for d in include_paths()]
    libs = [x for d in library_paths() for x in (f"-L{d}", f"-Wl,-rpath,{d}")]
    tmp = HOST_PATH + ".tmp"
    # NDEBUG: without it the headers bring a thread-local counter, and a library
    # with thread-local storage that no call touches keeps glibc's per-thread
    # table out of date: every thread-local access of the process (each torch
    # call makes some) then takes the slow lookup (torch.empty 1.07 -> 1.31 us,
    # Tensor.view 0.58 -> 0.66)
    _run(["g++", "-O2", "-DNDEBUG", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *inc, os.path.join(CSRC, "host.cpp"),
          "-o", tmp, *libs, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"])
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = False) -> str:
    """Compile every source and link the shared library and the extension that
    calls it; returns the library's path."""
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max_workers=1) as ex:
        host = ex.submit(_build_host)
        _build_lib(LIB_PATH, BUILD, [])
        host.result()
    # the microbenchmarks behind benchmarks/vector_rates.py, read_floor.py and prefill_step.py
    tools = [[HIPCC, *COMMON, "-x", "hip", os.path.join(PKG_DIR, "benchmarks", t + ".hip"), "-o", os.path.join(BUILD, t)]
             for t in BENCH_TOOLS]
    with ThreadPoolExecutor(max_workers=len(tools)) as ex:
        list(ex.map(_run, tools))
    if verbose:
        print(f"built {LIB_PATH}")
    return LIB_PATH


def build_timeline(verbose: bool = False) -> str:
    """The library once more with CIE_TIMELINE defined (per-workgroup stamps of
    the head-pair prefill and paged kernels, read by benchmarks/timeline.py);
    a measurement build, next to the product library, never loaded by it."""
    _build_lib(TIMELINE_LIB_PATH, os.path.join(BUILD, "timeline"), ["-DCIE_TIMELINE"])
    if verbose:
        print(f"built {TIMELINE_LIB_PATH}")
    return TIMELINE_LIB_PATH


if __name__ == "__main__":
    if "--timeline" in sys.argv[1:]:
        build_timeline(verbose=True)
    else:
        build(verbose=True)
