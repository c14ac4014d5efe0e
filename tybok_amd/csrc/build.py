"""Build libtybok_hip.so for gfx950 with plain hipcc (no torch headers), and the tk_calls extension, torch's side of its Python binding.

Run as ``python -m tybok_amd.csrc.build`` or through ``__graft_entry__.build()``.  hipcc
cross-compiles without a GPU; the library lands in ``tybok_amd/_lib/`` next to the package so it
travels with the source tree.  Each translation unit is compiled to an object of its own (in
parallel) and the objects are linked into the shared library.  tk_calls (host code only) is a CPython
extension that links against it; it is compiled for the Python that runs the build and that Python's torch
(the headers of both are needed) and has both in its file name.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

from .. import native

HERE = os.path.dirname(os.path.abspath(__file__))
LIB_DIR = os.path.join(os.path.dirname(HERE), "_lib")
OBJ_DIR = os.path.join(LIB_DIR, "obj")
LIB_PATH = os.path.join(LIB_DIR, "libtybok_hip.so")
CALLS_SOURCE = os.path.join(HERE, "tk_calls.cpp")
SOURCES = ("fp8w_gemm.hip", "fp8w_gemm_stream.hip", "fp8w_gemm_wide.hip", "expert_attn.hip", "expert_attn_d256.hip", "expert_attn_px.hip", "expert_tail.hip", "expert_kv_proj.hip", "layer_norm.hip", "tower_attn.hip", "rope_rows.hip", "prefix_prep.hip", "denoise_smolvla.hip", "denoise_pi05.hip", "stream_read.hip", "w8a8_gemm.hip", "bf16w_gemm_wide.hip", "tk_api.hip")
HEADERS = ("tk_common.h", "tk_kernels.h", "persist.h", "pipe_gemm.h", "pipe_fp8.h", os.path.join("..", "..", "include", "tybok_hip.h"))
ARCH = "gfx950"
FLAGS = (
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # keep hipcc from forming packed-fp32 VALU ops out of ordinary float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
)  # fmt: skip
_NOISE = "is not a recognized feature for this target"


def hipcc_path() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (looked on PATH and in /opt/rocm/bin)")


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print("[tybok_amd] " + " ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(line for line in proc.stderr.splitlines() if _NOISE not in line)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}): {' '.join(cmd)}\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)


def _calls_command(hipcc: str, out: str) -> list[str]:
    """The compile line of tk_calls; torch's libraries are in the process before it is loaded, so it names no path to them."""
    import torch

    root = os.path.dirname(torch.__file__)
    include, lib = os.path.join(root, "include"), os.path.join(root, "lib")
    return [
        hipcc, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM=1", "-D__HIP_PLATFORM_AMD__=1", f"-I{include}", f"-I{include}/torch/csrc/api/include",
        f"-I{os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(hipcc))), 'include')}", f"-I{sysconfig.get_paths()['include']}", CALLS_SOURCE, "-o", out, f"-L{lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip",
        f"-L{LIB_DIR}", "-ltybok_hip", "-Wl,-rpath,$ORIGIN",
    ]  # fmt: skip


def build_library(verbose: bool = True, incremental: bool = False, jobs: int = 8) -> str:
    """Compile every source and link the libraries.  ``incremental`` skips objects that are newer than
    their source and the shared headers (development convenience; the default compiles everything)."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    hipcc = hipcc_path()
    newest_header = max(os.path.getmtime(os.path.join(HERE, h)) for h in HEADERS)
    todo, objects = [], []
    for s in SOURCES:
        src = os.path.join(HERE, s)
        obj = os.path.join(OBJ_DIR, s.replace(".hip", ".o"))
        objects.append(obj)
        if incremental and os.path.exists(obj) and os.path.getmtime(obj) >= max(os.path.getmtime(src), newest_header):
            continue
        todo.append([hipcc, *FLAGS, "-c", src, "-o", obj])
    with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(todo) or 1))) as pool:
        list(pool.map(lambda cmd: _run(cmd, verbose), todo))
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,-soname,libtybok_hip.so", *objects, "-o", LIB_PATH + ".tmp"], verbose)
    os.replace(LIB_PATH + ".tmp", LIB_PATH)
    calls = native.calls_path()
    newest = max(os.path.getmtime(CALLS_SOURCE), os.path.getmtime(os.path.join(HERE, HEADERS[-1])))
    if not (incremental and os.path.exists(calls) and os.path.getmtime(calls) >= newest):
        _run(_calls_command(hipcc, calls + ".tmp"), verbose)
        os.replace(calls + ".tmp", calls)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(incremental="--incremental" in sys.argv))
