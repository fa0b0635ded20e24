"""Build recipe: ``libkdecay.so`` (one hipcc compilation per source for gfx950, then a link) and
``_native.so``, the host path of the Python functions (g++ against torch's headers).

Run ``python -m kilat_amd._build`` (or ``__graft_entry__.build()``).  The
library is written in-tree next to this file, where ``kilat_amd._lib`` loads it.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
SOURCES = [os.path.join(HERE, "csrc", name) for name in ("kdecay.hip", "kdecay_rows.hip")]
INCLUDE = os.path.join(ROOT, "include")
LIBRARY = os.path.join(HERE, "libkdecay.so")
NATIVE_SOURCE = os.path.join(HERE, "csrc", "native.cpp")
NATIVE = os.path.join(HERE, "_native.so")

# -packed-fp32-ops: no v_pk_*_f32 in the device code.
# -mcode-object-version=5: loadable by torch's bundled ROCm 7.0 runtime.
# No fast-math: fp32 division stays correctly rounded (hipcc's default), and
# the source turns fp contraction off itself.
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found (ROCm is required to build libkdecay.so)")
    return path


def build_library(verbose: bool = False) -> str:
    """Compile the csrc sources into libkdecay.so; returns the library path."""
    with tempfile.TemporaryDirectory(prefix="kdecay_build_") as work:
        jobs = []  # the sources compile side by side
        for src in SOURCES:
            obj = os.path.join(work, os.path.basename(src) + ".o")
            cmd = [hipcc(), *HIPCC_FLAGS, "-I", INCLUDE, "-c", src, "-o", obj]
            if verbose:
                print(" ".join(cmd), flush=True)
            jobs.append((obj, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        done = [(obj, proc.communicate()[0], proc.returncode) for obj, proc in jobs]
        tmp = LIBRARY + ".tmp"
        if all(rc == 0 for _, _, rc in done):
            cmd = [hipcc(), "--offload-arch=gfx950", "-shared", *[obj for obj, _, _ in done], "-o", tmp]
            if verbose:
                print(" ".join(cmd), flush=True)
            proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
            done.append((tmp, proc.stdout, proc.returncode))
        # hipcc's host pass does not know the packed-fp32 target feature and says
        # so; that line is expected and not shown.
        lines = [l for _, out, _ in done for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip()]
        if any(rc != 0 for _, _, rc in done):
            raise RuntimeError("hipcc failed:\n" + "\n".join(lines))
        if verbose and lines:
            print("\n".join(lines), flush=True)
        os.replace(tmp, LIBRARY)
    return LIBRARY


def build_native(verbose: bool = False) -> str:
    """Compile csrc/native.cpp into _native.so (after libkdecay.so, which it links); returns its path."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    tmp = NATIVE + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE]
    for path in [*cpp_extension.include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]:
        cmd += ["-isystem", path]
    cmd += [NATIVE_SOURCE, "-o", tmp, "-L", HERE, "-lkdecay", "-Wl,-rpath,$ORIGIN"]
    for path in cpp_extension.library_paths():
        cmd += ["-L", path]
    cmd += ["-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError("g++ failed:\n" + proc.stdout)
    if verbose and proc.stdout.strip():
        print(proc.stdout, flush=True)
    os.replace(tmp, NATIVE)
    return NATIVE


def build(verbose: bool = False) -> None:
    build_library(verbose)
    build_native(verbose)


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print(LIBRARY, NATIVE)
