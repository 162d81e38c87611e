"""Ahead-of-time build of the HIP kernels into ``ssm_amd/lib/libssm_amd.so``.

Run as ``python -m ssm_amd.build``.  The library exposes only the C ABI of
``include/ssm_amd.h``; it does not link against torch.

A second library, ``libssm_amd_testhooks.so``, is linked from the same objects
except that the sources which pick between kernels are compiled once more with
``-DSSM_TEST_HOOKS`` (``include/ssm_amd_testing.h``): the test suite uses it to
run a chosen kernel where the shipped library would pick another.

A third, ``_host.so``, is a Python extension module (C++ against torch, no device code): the host path of repeated
operator calls (``csrc/host/host.cpp``).  It calls the C ABI of whichever library ``ssm_amd._lib`` binds it to.
"""

from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OBJ = PKG / "lib" / "obj"
LIB = PKG / "lib" / "libssm_amd.so"
HOOKS_LIB = PKG / "lib" / "libssm_amd_testhooks.so"
HOST_SRC = CSRC / "host" / "host.cpp"
HOST_LIB = PKG / "lib" / "_host.so"
# the sources that read a kernel selector (SSM_RESERVED) or record the kernel taken
HOOKED = ("scan_fwd.hip", "scan_bwd.hip", "dscan_bwd.hip", "ssd.hip")

ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    # packed fp32 VALU forms are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unknown-cuda-version",
]


def hipcc() -> str:
    return os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _compile(src: Path, extra: list[str], suffix: str = "") -> Path:
    obj = OBJ / (src.stem + suffix + ".o")
    cmd = [hipcc(), *FLAGS, *extra, "-c", str(src), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _build_host() -> None:
    """The extension module of the host path; plain C++, so the host compiler builds it."""
    from torch.utils import cpp_extension

    rocm = Path(hipcc()).resolve().parent.parent
    inc = [*cpp_extension.include_paths(), sysconfig.get_paths()["include"],
           next(str(d) for d in (rocm / "include", Path("/opt/rocm/include")) if (d / "hip").is_dir())]
    libs = cpp_extension.library_paths()
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", *(f"-I{d}" for d in inc), str(HOST_SRC), "-o", str(HOST_LIB), *(f"-L{d}" for d in libs),
           "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", *(f"-Wl,-rpath,{d}" for d in libs)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on {HOST_SRC.name}:\n{proc.stderr}")


def build(verbose: bool = True, extra: list[str] | None = None, jobs: int | None = None) -> Path:
    """Compile every ``csrc/*.hip`` for gfx950, link the shared libraries, and build the host path's module."""
    OBJ.mkdir(parents=True, exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError("no HIP sources found")
    jobs = jobs or min(8, len(srcs))
    extra = extra or []
    hooked = [s for s in srcs if s.name in HOOKED]
    tasks = [(s, extra, "") for s in srcs] + [(s, [*extra, "-DSSM_TEST_HOOKS"], "_hooks") for s in hooked]
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_build_host)
        done = list(pool.map(lambda t: _compile(*t), tasks))
        host.result()
    objs, hook_objs = done[:len(srcs)], dict(zip((s.name for s in hooked), done[len(srcs):]))
    for lib, parts in ((LIB, objs), (HOOKS_LIB, [hook_objs.get(s.name, o) for s, o in zip(srcs, objs)])):
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(lib), *map(str, parts)]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed:\n{proc.stderr}")
    if verbose:
        print(f"built {LIB}, {HOOKS_LIB.name} and {HOST_LIB.name} from {len(srcs) + 1} sources")
    return LIB


if __name__ == "__main__":
    build(extra=sys.argv[1:])
