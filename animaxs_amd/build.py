"""Build libanima_hip.so in-tree with hipcc for gfx950.

``python -m animaxs_amd.build`` (or ``animaxs_amd.build.build()``) compiles every
``csrc/*.hip`` with ``hipcc --offload-arch=gfx950`` and every ``csrc/*.cpp`` with
``g++``, then links ``animaxs_amd/libanima_hip.so``; ``csrc/python/calls.cpp`` becomes the
CPython module ``animaxs_amd/_calls`` under the interpreter's own extension suffix, so that
another interpreter does not load it.  Packed-FP32 instruction selection is disabled for all
device code.
"""

from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
INCLUDE = ROOT / "include"
OUT = PKG / "libanima_hip.so"
CALLS = PKG / ("_calls" + sysconfig.get_config_var("EXT_SUFFIX"))
OBJ = PKG / "_build"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
HIP_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    f"-I{INCLUDE}", f"-I{CSRC}",
]
CXX_FLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", f"-I{INCLUDE}", f"-I{CSRC}"]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")


def _compile(src: Path) -> Path:
    obj = OBJ / (src.name + ".o")
    if src.suffix == ".hip":
        _run([HIPCC, "-x", "hip", "-c", str(src), "-o", str(obj), *HIP_FLAGS])
    else:
        _run([shutil.which("g++") or "g++", "-c", str(src), "-o", str(obj), *CXX_FLAGS])
    return obj


def _build_calls() -> None:
    tmp = CALLS.with_name(CALLS.name + ".tmp")
    _run([shutil.which("g++") or "g++", "-shared", str(CSRC / "python" / "calls.cpp"), "-o", str(tmp), *CXX_FLAGS,
          f"-I{sysconfig.get_paths()['include']}"])
    os.replace(tmp, CALLS)
    (PKG / "_calls.so").unlink(missing_ok=True)   # any interpreter would load an untagged one


def build(verbose: bool = True, jobs: int | None = None) -> Path:
    """Compile all sources and link the shared library; returns its path."""
    OBJ.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip")) + sorted(CSRC.glob("*.cpp"))
    if not sources:
        raise RuntimeError(f"no sources in {CSRC}")
    jobs = jobs or min(8, len(sources), os.cpu_count() or 4)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        calls = ex.submit(_build_calls)
        objs = list(ex.map(_compile, sources))
        calls.result()
    tmp = OUT.with_suffix(".so.tmp")
    _run([HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", str(tmp), *map(str, objs)])
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT} ({OUT.stat().st_size} bytes) from {len(sources)} sources")
    return OUT


if __name__ == "__main__":
    build()
    sys.exit(0)
