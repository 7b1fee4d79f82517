"""Build of the native library ``aklr_amd/libaklr_amd.so`` from ``aklr_amd/csrc/*.hip`` with hipcc.

In-tree build for gfx950 only: every ``.hip`` file compiles to an object in ``aklr_amd/_build/`` (in
parallel), then hipcc links them into one shared library exporting the C ABI of
``include/aklr_amd.h``. Mirrors the role of aklr/core/jit/hip_extension.py (hipcc, ``-O3``, one arch),
without torch in the loop: the library has no torch types in its interface. ``aklr_amd/_host.*.so``
(``csrc/host/host.cpp``) is the one part that has them: the ops' host work as a Python extension, built
with the host compiler against torch's headers and linked to the library beside it. It refuses another
torch version than the one it was built with.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD_DIR = PKG / "_build"
LIB_PATH = PKG / "libaklr_amd.so"
HOST_SRC = CSRC / "host" / "host.cpp"
HOST_PATH = PKG / f"_host{sysconfig.get_config_var('EXT_SUFFIX')}"  # no other Python imports it
ARCH = "gfx950"

# Packed-fp32 VALU ops are switched off: the kernels' fp32 arithmetic stays scalar per lane. The sources
# also switch them off themselves (AKLR_SCALAR_FP32_BEGIN/END), for builds that pass no such flag.
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-fPIC",
    "-std=c++17",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the aklr_amd native library needs ROCm's hipcc to build")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(src: Path) -> Path:
    obj = BUILD_DIR / (src.stem + ".o")
    cmd = [hipcc(), *HIP_FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stderr}")
    return obj


def _link_host() -> None:
    """``_host.*.so``: it finds ``libaklr_amd.so`` by its run path, torch's libraries by the process."""
    import torch

    root = Path(torch.__file__).resolve().parent
    rocm = Path(hipcc()).resolve().parent.parent
    if not (rocm / "include" / "hip").is_dir():
        rocm = Path("/opt/rocm")
    tmp = HOST_PATH.with_suffix(".so.tmp")
    cmd = [
        os.environ.get("CXX") or "g++", "-O2", "-fPIC", "-shared", "-std=c++17", "-D__HIP_PLATFORM_AMD__=1",
        "-DUSE_ROCM=1", f'-DAKLR_TORCH_VERSION="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f"-I{root}/include",
        f"-I{root}/include/torch/csrc/api/include", f"-I{rocm}/include", f"-I{sysconfig.get_paths()['include']}",
        str(HOST_SRC), "-o", str(tmp), f"-L{root}/lib", "-ltorch_python", "-ltorch_cpu", "-ltorch_hip", "-ltorch",
        "-lc10_hip", "-lc10", f"-L{PKG}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN",
    ]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"building {HOST_PATH.name} failed:\n{res.stderr}")
    os.replace(tmp, HOST_PATH)


def build(verbose: bool = False) -> Path:
    """Compile every kernel source, link ``libaklr_amd.so`` and build ``_host.*.so`` on it; returns the
    library's path."""
    BUILD_DIR.mkdir(exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    workers = min(len(srcs), max(1, (os.cpu_count() or 4) // 2), 8)
    with concurrent.futures.ThreadPoolExecutor(max_workers=workers) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc link failed:\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host()
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources")
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
