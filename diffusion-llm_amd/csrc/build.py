"""Build libbd3attn.so for gfx950 with hipcc (no GPU needed: hipcc
cross-compiles the device code) and bd3_host.so, the CPython extension that
prepares the kernels' calls, with g++ against the installed torch.

    python diffusion-llm_amd/csrc/build.py [--jobs N] [--verbose]

Sources: every *.hip file in this directory, and host_calls.cpp. Output:
diffusion-llm_amd/lib/libbd3attn.so and bd3_host.so (git-ignored).
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

CSRC = Path(__file__).resolve().parent
PKG = CSRC.parent
REPO = PKG.parent
LIB_DIR = PKG / "lib"
LIB = LIB_DIR / "libbd3attn.so"
HOST = LIB_DIR / "bd3_host.so"
OBJ_DIR = PKG / "_build"

ARCH = "gfx950"

# -packed-fp32-ops: hipcc would otherwise fuse float pairs into
# v_pk_{add,mul,fma}_f32, some forms of which have given wrong results on gfx950.
# The host pass warns that it does not know the feature; that is harmless.
# -mno-amdgpu-ieee -fno-honor-nans: the kernels never produce or consume
# NaN (masked scores are -inf, every row has a live key), so the IEEE-mode
# NaN quieting the compiler would otherwise insert before each max (one
# extra v_max per softmax element) is dropped and max chains fold into
# v_max3_f32.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-munsafe-fp-atomics",
    "-mno-amdgpu-ieee",
    "-fno-honor-nans",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
    f"-I{REPO / 'include'}",
    f"-I{CSRC}",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found (ROCm toolchain required to build libbd3attn.so)")
    return path


def _compile(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in res.stderr.splitlines() if noise not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if verbose and err.strip():
        print(err, flush=True)
    return obj


def _build_host(verbose: bool) -> Path:
    """bd3_host.so: host code only, so g++ and torch's headers and libraries."""
    from torch.utils import cpp_extension
    torch_lib = Path(cpp_extension.include_paths()[0]).parent / "lib"
    rocm = Path(hipcc()).resolve().parent.parent
    tmp = HOST.with_suffix(".so.tmp")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wno-deprecated-declarations",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",  # what torch's HIP headers are compiled with
           str(CSRC / "host_calls.cpp"), "-o", str(tmp), f"-I{REPO / 'include'}",
           *(f"-I{p}" for p in cpp_extension.include_paths()), f"-I{rocm / 'include'}",
           f"-I{sysconfig.get_paths()['include']}", f"-L{torch_lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu",
           "-ltorch_hip", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on host_calls.cpp:\n{res.stderr}")
    os.replace(tmp, HOST)
    return HOST


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every .hip source, link libbd3attn.so and build bd3_host.so.
    Always rebuilds."""
    OBJ_DIR.mkdir(parents=True, exist_ok=True)
    LIB_DIR.mkdir(parents=True, exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no .hip sources in {CSRC}")
    jobs = jobs or min(len(sources), os.cpu_count() or 4, 8)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        host = ex.submit(_build_host, verbose)
        objs = list(ex.map(lambda s: _compile(s, verbose), sources))
        host.result()
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, LIB)
    return LIB


def main(argv: list[str] | None = None) -> int:
    p = argparse.ArgumentParser(description=__doc__)
    p.add_argument("--jobs", type=int, default=None)
    p.add_argument("--verbose", action="store_true")
    args = p.parse_args(argv)
    lib = build(args.jobs, args.verbose)
    print(f"built {lib}")
    return 0


if __name__ == "__main__":
    sys.exit(main())
