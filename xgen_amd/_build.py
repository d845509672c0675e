"""Builds the gfx950 HIP library libxgen_amd.so in-tree (hipcc, no torch headers) and the
torch operators' host library libxgen_amd_ops.so (g++, torch headers).

Each csrc/*.hip file is compiled to an object in parallel, then linked into
xgen_amd/_lib/libxgen_amd.so.  The library links libamdhip64.so.7; loaded after
`import torch`, it binds to the HIP runtime torch already loaded (same soname).
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
from pathlib import Path

PACKAGE = Path(__file__).resolve().parent
ROOT = PACKAGE.parent
CSRC = PACKAGE / "csrc"
INCLUDE = ROOT / "include"
OUT_DIR = PACKAGE / "_lib"
LIBRARY = OUT_DIR / "libxgen_amd.so"
OPERATORS = OUT_DIR / "libxgen_amd_ops.so"
OBJ_DIR = ROOT / "_build" / "xgen_amd"

ARCH = "gfx950"
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-mcode-object-version=5",
    "-Wall",
    "-Wno-unused-function",
    # packed fp32 VALU forms are disabled for every kernel in this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build xgen_amd")
    return path


def _compile(src: Path) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [hipcc(), *HIP_FLAGS, f"-I{INCLUDE}", f"-I{CSRC}", "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{proc.stdout}")
    return obj


def _operators() -> Path:
    """csrc/torch_ops.cpp: host code only; links torch, and opens libxgen_amd.so at run time."""
    import torch
    root = Path(torch.__file__).resolve().parent
    rocm = Path(hipcc()).resolve().parent.parent
    tmp = OPERATORS.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "c++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{INCLUDE}", "-isystem", str(root / "include"), "-isystem", str(root / "include/torch/csrc/api/include"),
           "-isystem", str(rocm / "include"), str(CSRC / "torch_ops.cpp"), "-o", str(tmp),
           f"-L{root / 'lib'}", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ldl"]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"g++ failed for torch_ops.cpp:\n{proc.stdout}")
    os.replace(tmp, OPERATORS)
    return OPERATORS


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compiles every csrc/*.hip for gfx950 and links libxgen_amd.so (returns its path), and the
    torch operators' library beside it."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    OUT_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(len(sources), max(1, (os.cpu_count() or 4)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs + 1) as pool:
        operators = pool.submit(_operators)
        objects = list(pool.map(_compile, sources))
        operators.result()
    tmp = LIBRARY.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)]
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{proc.stdout}")
    os.replace(tmp, LIBRARY)
    if verbose:
        print(f"built {LIBRARY}")
        print(f"built {OPERATORS}")
    return LIBRARY


if __name__ == "__main__":
    build(verbose=True)
