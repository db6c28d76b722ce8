"""Compile the gfx950 HIP sources into the in-tree C-ABI library librlt_kv.so,
and the host calls (host_calls.cpp) into the extension module beside it.

Every call recompiles (no up-to-date check): the caller decides when to build.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sysconfig
import warnings
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
PROJECT_DIR = PACKAGE_DIR.parent
REPO_DIR = PROJECT_DIR.parent
CSRC_DIR = PROJECT_DIR / "csrc"
INCLUDE_DIR = REPO_DIR / "include"
BUILD_DIR = PROJECT_DIR / "_build"
LIBRARY = PACKAGE_DIR / "librlt_kv.so"
HOST_CALLS = PACKAGE_DIR / "_host_calls.so"
ARCH = "gfx950"

# Packed-fp32 VALU forms are disabled for all device code; -O3 would otherwise
# emit v_pk_{add,mul,fma}_f32 from ordinary float code.
DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(path).exists():
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build librlt_kv.so")
    return path


def sources() -> list[Path]:
    return sorted(CSRC_DIR.glob("*.hip"))


def _compile(source: Path) -> Path:
    obj = BUILD_DIR / (source.stem + ".o")
    cmd = [hipcc(), *DEVICE_FLAGS, f"-I{INCLUDE_DIR}", f"-I{CSRC_DIR}", "-c", str(source), "-o", str(obj)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"hipcc failed on {source.name}:\n{result.stderr}")
    return obj


def build_host_calls() -> Path:
    """The Python extension of csrc/host_calls.cpp, against the installed torch."""
    import torch
    from torch.utils import cpp_extension

    includes = [INCLUDE_DIR, sysconfig.get_paths()["include"], *cpp_extension.include_paths()]
    tmp = HOST_CALLS.with_suffix(".so.tmp")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall"]
    cmd += [f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{i}" for i in includes)]
    cmd += [str(CSRC_DIR / "host_calls.cpp"), f"-L{Path(torch.__file__).parent / 'lib'}"]
    cmd += ["-ltorch_python", "-ltorch_cpu", "-lc10", "-o", str(tmp)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"g++ failed on host_calls.cpp:\n{result.stderr}")
    os.replace(tmp, HOST_CALLS)
    return HOST_CALLS


def build(jobs: int | None = None) -> Path:
    """Compile every csrc/*.hip for gfx950 and link librlt_kv.so in the package, beside its host calls.

    The library does without the host calls: where they cannot be built (they need
    g++, Python's and torch's headers) there are none, not even old ones, and a
    warning says so.
    """
    BUILD_DIR.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC_DIR}")
    jobs = jobs or min(len(srcs), max(1, (os.cpu_count() or 2) // 2), 8)
    with ThreadPoolExecutor(jobs) as pool:
        host_calls = pool.submit(build_host_calls)
        objects = list(pool.map(_compile, srcs))
        try:
            host_calls.result()
        except (RuntimeError, OSError, ImportError) as error:
            HOST_CALLS.unlink(missing_ok=True)
            warnings.warn(f"the C++ host calls were not built, calls will go through Python (slower): {error}", stacklevel=2)
    tmp = LIBRARY.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)]
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        raise RuntimeError(f"linking librlt_kv.so failed:\n{result.stderr}")
    os.replace(tmp, LIBRARY)
    return LIBRARY


if __name__ == "__main__":
    print(build())
