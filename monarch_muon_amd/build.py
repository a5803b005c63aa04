"""Build ``libmmuon.so`` (gfx950) in-tree with hipcc.

``python -m monarch_muon_amd.build`` compiles every ``csrc/*.hip`` to an object
in parallel and links the shared library next to this file, and beside it
``libmmuon_torch.<ABI>.so``, the layer's native torch operator (``csrc/torch_ops.cpp``,
host code only).  hipcc cross-compiles for gfx950 without a GPU.  ``build_probe()`` builds the
bench-only HBM streaming probe (``bench_probe.hip`` beside ``bench.py``) into a
library of its own, apart from the optimizer's.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
from pathlib import Path

from ._abi import TORCH_LIB_PATH as TORCH_LIB

HERE = Path(__file__).resolve().parent
CSRC = HERE / "csrc"
LIB = HERE / "libmmuon.so"
ARCH = "gfx950"

CFLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # every rounding the reference performs is explicit; no silent FMA contraction
    "-ffp-contract=off",
    # packed fp32 VALU ops are disabled for every kernel
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build libmmuon.so")
    return exe


def _compile(src: Path, obj: Path) -> None:
    cmd = [_hipcc(), *CFLAGS, "-c", str(src), "-o", str(obj)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        msg = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
        raise RuntimeError(f"hipcc failed on {src.name}:\n{msg}")


def _build_torch_ops() -> None:
    import torch
    inc = Path(torch.__file__).resolve().parent
    rocm = Path(_hipcc()).resolve().parent.parent
    tmp = TORCH_LIB.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-isystem", str(inc / "include"), "-isystem", str(inc / "include/torch/csrc/api/include"),
           "-isystem", str(rocm / "include"), "-isystem", "/opt/rocm/include", str(CSRC / "torch_ops.cpp"),
           "-o", str(tmp), f"-L{inc / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"torch_ops.cpp failed:\n{r.stdout}{r.stderr}")
    os.replace(tmp, TORCH_LIB)
    for old in HERE.glob("libmmuon_torch*.so"):   # built for another ABI: never loaded again
        if old != TORCH_LIB:
            old.unlink()


def build(verbose: bool = True) -> Path:
    srcs = sorted(CSRC.glob("*.hip"))
    objdir = HERE / "_build"
    objdir.mkdir(exist_ok=True)
    objs = [objdir / (s.stem + ".o") for s in srcs]
    jobs = max(1, min(len(srcs), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4))))
    with cf.ThreadPoolExecutor(jobs + 1) as ex:
        ops = ex.submit(_build_torch_ops)
        list(ex.map(_compile, srcs, objs))
        ops.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources", file=sys.stderr)
    return LIB


def build_probe(verbose: bool = True) -> Path:
    """``bench_probe.so`` from ``bench_probe.hip`` at the repository root (used
    only by ``bench.py --hbm-ceiling`` / ``--data-energy``)."""
    root = HERE.parent
    src, out = root / "bench_probe.hip", root / "bench_probe.so"
    tmp = out.with_suffix(".so.tmp")
    cmd = [_hipcc(), *CFLAGS, "-shared", f"-I{root}", str(src), "-o", str(tmp)]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        msg = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
        raise RuntimeError(f"hipcc failed on {src.name}:\n{msg}")
    os.replace(tmp, out)
    if verbose:
        print(f"built {out}", file=sys.stderr)
    return out


if __name__ == "__main__":
    build()
