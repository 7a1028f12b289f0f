"""Build libhdcmamba_hip.so in-tree for gfx950 with hipcc.

Usage:  python -m hdcmamba_amd.build        (or hdcmamba_amd.build.build())

Every csrc/*.hip file is compiled to an object under hdcmamba_amd/_build/ and the
objects are linked into hdcmamba_amd/libhdcmamba_hip.so, which is what
hdcmamba_amd._ops loads.  Packed-fp32 VALU ops are disabled for device code.
csrc/native.cpp (host code over PyTorch's C++ API) is compiled with g++ into the extension
module hdcmamba_amd/_native.so, linked against that library.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB = PKG / "libhdcmamba_hip.so"
NATIVE = PKG / "_native.so"
ARCH = os.environ.get("HDCM_OFFLOAD_ARCH", "gfx950")

CFLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-Wall",
    "-Wno-unused-function", "-Wno-unused-variable",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found (ROCm is required to build libhdcmamba_hip.so)")


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    # The host pass does not know the device-only target feature; drop that one warning.
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops' is not a recognized" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{err}")
    return err


def _compile_native() -> str:
    """csrc/native.cpp to an object, against the running interpreter's torch and Python headers."""
    import sysconfig

    from torch.utils import cpp_extension

    inc = [str(PKG.parent / "include"), *cpp_extension.include_paths(), sysconfig.get_paths()["include"]]
    return _run(["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-DTORCH_EXTENSION_NAME=_native",
                 "-DTORCH_API_INCLUDE_EXTENSION_H", *[f"-I{p}" for p in inc], "-c", str(CSRC / "native.cpp"), "-o",
                 str(BUILD / "native.o")])


def _link_native() -> None:
    import torch

    lib = str(Path(torch.__file__).parent / "lib")
    tmp = NATIVE.with_suffix(".so.tmp")
    _run(["g++", "-shared", str(BUILD / "native.o"), "-o", str(tmp), f"-L{PKG}", "-l:libhdcmamba_hip.so", f"-L{lib}",
          "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN", f"-Wl,-rpath,{lib}"])
    os.replace(tmp, NATIVE)


def build(verbose: bool = False) -> Path:
    hipcc = _hipcc()
    BUILD.mkdir(exist_ok=True)
    srcs = sorted(CSRC.glob("*.hip"))
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    objs = [BUILD / (s.stem + ".o") for s in srcs]
    jobs = min(len(srcs), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        native = ex.submit(_compile_native)
        futs = [ex.submit(_run, [hipcc, *CFLAGS, "-I", str(PKG.parent / "include"), "-c", str(s), "-o", str(o)])
                for s, o in zip(srcs, objs)]
        for s, f in zip(srcs, futs):
            msg = f.result()
            if verbose and msg.strip():
                print(f"[{s.name}]\n{msg}", file=sys.stderr)
        msg = native.result()
        if verbose and msg.strip():
            print(f"[native.cpp]\n{msg}", file=sys.stderr)
    tmp = LIB.with_suffix(".so.tmp")
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)])
    os.replace(tmp, LIB)
    _link_native()
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
