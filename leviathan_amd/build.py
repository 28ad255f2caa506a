"""Builds ``libleviathan_hip.so`` (gfx950 only) from ``csrc/*.hip`` with hipcc, and with the host compiler
``_lev_ops.so``, the argument handling of ``ops.py``, from ``csrc/py_ops.cpp``.

Run ``python -m leviathan_amd.build``.  hipcc cross-compiles without a GPU.  Without torch or a host compiler
the library alone is built.
Objects are compiled in parallel and linked into ``leviathan_amd/lib``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
OBJ_DIR = os.path.join(HERE, "build")
LIB_PATH = os.path.join(LIB_DIR, "libleviathan_hip.so")
OPS_PATH = os.path.join(LIB_DIR, "_lev_ops.so")

ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-warning-option",
    # packed FP32 VALU ops are not to be generated for this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# The first 16 dwords of plain kernel arguments arrive in registers with the wave: a trip to memory less in front of the first
# requests.  us without and with it: the Q4_0 GEMV of 4096 x 4096 on cold weights 3.85 and 3.63; among other calls RMSNorm and Q4_K by
# four columns (12288 x 4096) 9.1 and 8.8, the int8 FFN of five columns (4096 / 12288) 31.8 and 31.0, 64 tokens through an MoE layer
# (2048 / 768) 95.5 and 94.0.  Recorded kernels of few us on weights that the caches hold lose up to 2 %: that GEMV 3.21 and 3.27,
# Q4_K by two columns (4096 x 4096) 5.55 and 5.63, the int8 FFN of one column (1024 / 2048) 14.77 and 14.96.
# Not for the Q6_K head's long stream, which takes 105.3 us with it and 104.3 without.
PRELOAD_FLAGS = ["-mllvm", "-amdgpu-kernarg-preload-count=16"]
NO_PRELOAD = {"q6_k_mfma_gemv.hip"}


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found")
    return exe


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _headers_mtime() -> float:
    paths = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hpp")]
    paths.append(os.path.join(HERE, "..", "include", "leviathan_hip.h"))
    return max(os.path.getmtime(p) for p in paths)


def _compile(src: str, force: bool, extra: list[str]) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    preload = [] if os.path.basename(src) in NO_PRELOAD else PRELOAD_FLAGS
    cmd = [hipcc(), *HIPCC_FLAGS, *preload, *extra, "-c", src, "-o", obj]
    made_by = obj + ".cmd"                   # an object made by another command is not up to date
    if (not force and os.path.exists(obj) and os.path.exists(made_by) and open(made_by).read() == "\n".join(cmd)
            and os.path.getmtime(obj) >= max(os.path.getmtime(src), _headers_mtime())):
        return obj
    if os.path.exists(made_by):
        os.remove(made_by)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l and l.strip())
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err:
        sys.stderr.write(err + "\n")
    with open(made_by, "w") as f:
        f.write("\n".join(cmd))
    return obj


def _build_ops(force: bool) -> str:
    """The CPython extension. It names torch's libraries without a path: they are loaded when it is.

    Returns what it lacks where torch or a host compiler is missing, which only ``ops.py`` needs: the C library and
    its callers do without.
    """
    import sysconfig
    try:
        from torch.utils import cpp_extension
    except ImportError:
        return "torch"
    src = os.path.join(CSRC, "py_ops.cpp")
    if (not force and os.path.exists(OPS_PATH)
            and os.path.getmtime(OPS_PATH) >= max(os.path.getmtime(src), _headers_mtime())):
        return ""
    cxx = shutil.which(os.environ.get("CXX") or "g++")
    if not cxx:
        return "a C++ compiler (g++, or the one CXX names)"
    tmp = OPS_PATH + ".tmp"
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden",
           *(a for p in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"]) for a in ("-isystem", p)),
           src, "-o", tmp, f"-L{LIB_DIR}", *(f"-L{p}" for p in cpp_extension.library_paths()),
           "-lleviathan_hip", "-ltorch_python", "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for {src}:\n{res.stderr}")
    os.replace(tmp, OPS_PATH)
    return ""


def build(force: bool = True, jobs: int = 8, extra_flags: list[str] | None = None) -> str:
    os.makedirs(LIB_DIR, exist_ok=True)
    os.makedirs(OBJ_DIR, exist_ok=True)
    extra = list(extra_flags or [])
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        objs = list(pool.map(lambda s: _compile(s, force, extra), sources()))
    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    lacks = _build_ops(force)
    if lacks:
        sys.stderr.write(f"{os.path.basename(OPS_PATH)}, which leviathan_amd.ops loads, is not built: it needs {lacks}\n")
    return LIB_PATH


if __name__ == "__main__":
    incremental = "--incremental" in sys.argv
    print(build(force=not incremental))
