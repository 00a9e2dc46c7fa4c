"""Build libqgemm.so (gfx950) and _fast.so in-tree.

Every ``csrc/*.hip`` file is compiled to an object under ``_build/`` (in
parallel) and linked into ``libqgemm.so`` next to this file.  All HIP code is
compiled with packed-FP32 instruction generation disabled.  ``csrc/host/fast.cpp``
(host code against torch's headers: the Python wrappers' plain calls) becomes
``_fast.so``; where it cannot be built (no torch, no g++) a warning says so, and
the wrappers make those calls in Python.
"""
import os
import subprocess
import sys
import warnings
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
OUT_DIR = PKG / "_build"
LIB = PKG / "libqgemm.so"
FAST = PKG / "_fast.so"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

HIPFLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", str(ROOT / "include"),
    "-I", str(CSRC),
]


def _compile(src: Path) -> Path:
    obj = OUT_DIR / (src.stem + ".o")
    cmd = [HIPCC, *HIPFLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr}")
    return obj


def _build_fast() -> None:
    FAST.unlink(missing_ok=True)    # never one of an older library
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    torch_lib = Path(torch.__file__).resolve().parent / "lib"
    tmp = FAST.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-I", str(ROOT / "include"),
           "-I", sysconfig.get_paths()["include"],
           *[f for d in cpp_extension.include_paths("cuda") for f in ("-isystem", d)],
           str(CSRC / "host" / "fast.cpp"), "-o", str(tmp), "-L", str(torch_lib),
           "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for fast.cpp:\n{res.stderr}")
    os.replace(tmp, FAST)


def build(jobs: int = 8, verbose: bool = False) -> Path:
    OUT_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(sources)))) as ex:
        fast = ex.submit(_build_fast)
        objs = list(ex.map(_compile, sources))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    if fast.exception():
        warnings.warn(f"{FAST.name} was not built, calls go through Python: {fast.exception()}")
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
