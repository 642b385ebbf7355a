"""Builds libtorsh_hipq.so (the C-ABI library) for gfx950 with hipcc, and the module that carries Python's calls into it.

Run as ``python -m torsh_amd.build``.  hipcc cross-compiles, so no GPU is
needed to build.  Objects are compiled in parallel and linked in-tree at
``torsh_amd/lib/libtorsh_hipq.so``.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OBJ_DIR = os.path.join(PKG, "lib", "obj")
LIB_PATH = os.path.join(PKG, "lib", "libtorsh_hipq.so")
PYTHON_PATH = os.path.join(PKG, "lib", "_hipq_python.so")
PYTHON_STAMP = os.path.join(OBJ_DIR, "_hipq_python.stamp")  # what the module was built against

ARCH = "gfx950"

# -ffp-contract=off and the correctly rounded divide keep every f32 operation an
# individually rounded IEEE operation (bit parity with the CPU reference path);
# packed-fp32 instructions are switched off for the device pass.
HIPCC_FLAGS = [
    "-O3",
    "-std=c++17",
    f"--offload-arch={ARCH}",
    "-fPIC",
    "-fvisibility=hidden",
    "-ffp-contract=off",
    "-fno-fast-math",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-command-line-argument",
    "-I", os.path.join(ROOT, "include"),
    "-I", CSRC,
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the HIP toolchain is required to build torsh_hipq")
    return exe


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _headers_mtime() -> float:
    paths = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    paths.append(os.path.join(ROOT, "include", "torsh_hipq.h"))
    return max(os.path.getmtime(p) for p in paths)


def _compile(src: str, force: bool) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    if not force and os.path.exists(obj):
        if os.path.getmtime(obj) >= max(os.path.getmtime(src), _headers_mtime()):
            return obj
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{proc.stdout}\n{proc.stderr}")
    warn = "\n".join(l for l in proc.stderr.splitlines() if "packed-fp32-ops" not in l and l.strip())
    if warn:
        sys.stderr.write(warn + "\n")
    return obj


def _build_python(force: bool) -> None:
    """The Python side of the library's calls (csrc/hipq_python.cpp), host code against torch's headers."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    src = os.path.join(CSRC, "hipq_python.cpp")
    newest = max(os.path.getmtime(src), os.path.getmtime(os.path.join(ROOT, "include", "torsh_hipq.h")))
    against = f"python {sys.version}\ntorch {torch.__version__} {torch.__file__}\n"
    if not force and os.path.exists(PYTHON_PATH) and os.path.getmtime(PYTHON_PATH) >= newest and os.path.exists(PYTHON_STAMP):
        with open(PYTHON_STAMP) as f:
            if f.read() == against:
                return
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", os.path.join(ROOT, "include"),
           "-isystem", sysconfig.get_paths()["include"]]
    for path in cpp_extension.include_paths():
        cmd += ["-isystem", path]
    cmd += [src, "-o", PYTHON_PATH, "-L", os.path.dirname(LIB_PATH), "-l:libtorsh_hipq.so", "-Wl,-rpath,$ORIGIN"]
    for path in cpp_extension.library_paths():
        cmd += ["-L", path]
    cmd += ["-ltorch_python", "-ltorch_cpu", "-lc10"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"building {src} failed:\n{proc.stdout}\n{proc.stderr}")
    with open(PYTHON_STAMP, "w") as f:
        f.write(against)


def build(force: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=max(1, min(jobs, len(srcs)))) as pool:
        objs = list(pool.map(lambda s: _compile(s, force), srcs))
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", LIB_PATH, *objs]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}\n{proc.stderr}")
    _build_python(force)
    return LIB_PATH


if __name__ == "__main__":
    incremental = "--incremental" in sys.argv
    print(build(force=not incremental))
