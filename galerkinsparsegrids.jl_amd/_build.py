"""Build libgsg.so (gfx950) in-tree with hipcc.

Every HIP translation unit is compiled with packed-FP32 instructions disabled
(`-Xclang -target-feature -Xclang -packed-fp32-ops`).
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
OBJ = PKG / "_obj"
LIB = PKG / "libgsg.so"

ARCH = os.environ.get("GSG_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function", f"-I{ROOT / 'include'}", f"-I{CSRC}"]
HIPFLAGS = [f"--offload-arch={ARCH}", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]

# (source, HIP, part): a source with parts is compiled once per part (GSG_PART), the
# parts side by side
SOURCES = [
    ("gsg_setup.cpp", False, None),
    ("gsg_capi.cpp", True, None),
    ("gsg_kernels.hip", True, 0),
    ("gsg_kernels.hip", True, 1),
    ("gsg_kernels.hip", True, 2),
    ("gsg_kernels.hip", True, 3),
    ("gsg_kernels.hip", True, 4),
    ("gsg_solo64.hip", True, None),
    ("gsg_solo32.hip", True, None),
]


def _object(src: str, part) -> Path:
    return OBJ / (Path(src).stem + ("" if part is None else f"_{part}") + ".o")


def _compile(src: str, hip: bool, part, verbose: bool) -> Path:
    out = _object(src, part)
    cmd = [HIPCC] + COMMON + (HIPFLAGS if hip else ["-x", "c++"]) + ["-c", str(CSRC / src), "-o", str(out)]
    if part is not None:
        cmd.insert(-4, f"-DGSG_PART={part}")
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    if verbose and r.stderr.strip():
        print(r.stderr, file=sys.stderr)
    return out


def build(verbose: bool = False) -> Path:
    """Compile every source and link libgsg.so next to this file."""
    OBJ.mkdir(exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(len(SOURCES), os.cpu_count() or 1)) as ex:
        objs = list(ex.map(lambda s: _compile(*s, verbose), SOURCES))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp)] + [str(o) for o in objs] + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
