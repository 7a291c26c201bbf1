"""Builds libflashmaxsim.so (the HIP kernels + C ABI) in-tree for gfx950.

Usage: ``python -m flash_maxsim_amd.build`` or ``flash_maxsim_amd.build.build()``.
Every ``csrc/*.hip`` file is compiled to an object with hipcc (in parallel),
then linked into ``flash_maxsim_amd/libflashmaxsim.so`` next to this file;
``csrc/native.cpp``, the host path of the ordinary calls, is compiled with the
host compiler against torch's headers into ``flash_maxsim_amd/_native.so``,
which links to that library.
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
OBJ_DIR = PKG_DIR / "_build"
LIB_PATH = PKG_DIR / "libflashmaxsim.so"
NATIVE_PATH = PKG_DIR / "_native.so"

ARCH = os.environ.get("FMX_OFFLOAD_ARCH", "gfx950")

# Packed fp32 VALU ops are disabled: hand-rolled or compiler-formed
# v_pk_{add,mul,fma}_f32 are not used anywhere in this library.
# MFMAs accumulate in VGPRs (gfx950's unified register file) rather than AGPRs:
# the epilogues read every result, and the AGPR form costs a v_accvgpr_read
# per result register.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-mllvm",
    "-amdgpu-mfma-vgpr-form",
]


def _hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found: the ROCm toolchain is required to build libflashmaxsim")
    return path


def _compile(src: Path, verbose: bool) -> Path:
    obj = OBJ_DIR / (src.stem + ".o")
    cmd = [_hipcc(), *HIP_FLAGS, "-c", str(src), "-o", str(obj)]
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stdout}\n{res.stderr}")
    return obj


def _run(cmd: list[str], what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stdout}\n{res.stderr}")


def _compile_native(verbose: bool) -> Path:
    from torch.utils.cpp_extension import include_paths

    obj = OBJ_DIR / "native.o"
    dirs = [*include_paths(device_type="cuda"), sysconfig.get_paths()["include"]]
    # NDEBUG, as torch itself: without it pybind11's headers define a thread-local
    # counter. Once a library with thread-local storage is loaded, glibc (2.35) takes
    # its slow way for the thread-local variables of all libraries loaded before it,
    # torch's among them, in every thread that has not used the new one's, and nothing
    # here uses that counter: an add of two small GPU tensors took 5.3 us instead of
    # 4.4, topk_scores of 10 x 500 12.0 instead of 10.5.
    _run(["g++", "-std=c++17", "-O2", "-DNDEBUG", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          *(f"-isystem{d}" for d in dirs), "-c", str(CSRC / "native.cpp"), "-o", str(obj)], "g++ on native.cpp", verbose)
    return obj


def _link_native(obj: Path, verbose: bool) -> None:
    from torch.utils.cpp_extension import library_paths

    tmp = NATIVE_PATH.with_suffix(".so.tmp")
    _run(["g++", "-shared", str(obj), "-o", str(tmp), f"-L{PKG_DIR}", "-lflashmaxsim",
          *(f"-L{d}" for d in library_paths(device_type="cuda")), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10",
          "-lc10_hip", "-Wl,-rpath,$ORIGIN"], "link of _native.so", verbose)
    os.replace(tmp, NATIVE_PATH)


def build(verbose: bool = False, jobs: int | None = None) -> Path:
    """Compiles every source, links libflashmaxsim.so and _native.so; returns the library's path."""
    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    jobs = jobs or min(len(sources), max(1, (os.cpu_count() or 2)))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        native = pool.submit(_compile_native, verbose)
        objs = list(pool.map(lambda s: _compile(s, verbose), sources))
        native_obj = native.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    _run(cmd, "link", verbose)
    os.replace(tmp, LIB_PATH)
    _link_native(native_obj, verbose)
    return LIB_PATH


if __name__ == "__main__":
    out = build(verbose="-v" in sys.argv)
    print(out)
