"""Build liblinquant_hip.so (all HIP kernels + the C ABI) for gfx950 with hipcc, and the wrappers' native host code.

``python -m linquant_amd.build`` compiles in-tree; the library lands next to the sources so it travels with
the repository snapshot.  hipcc cross-compiles without a GPU.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

CSRC = Path(__file__).resolve().parent / "csrc"
LIB_PATH = CSRC / "liblinquant_hip.so"
BINDING_PATH = CSRC.parent / "_binding.so"
ARCH = "gfx950"

# -ffp-contract=off: every fp32 multiply/add that feeds an INT8 code is rounded on its own (the CPU checker
# restates the same sequences); the packed-fp32 feature is switched off for the device pass.
FLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-ffp-contract=off",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops", "-Wno-unused-command-line-argument"]


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found: the HIP kernels cannot be built")
    return exe


def _compile(src: Path, obj: Path) -> None:
    cmd = [_hipcc(), *FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stderr}")


def built_for() -> str:
    """What binding.cpp is compiled against besides its own sources: torch's and Python's binary interfaces.  The compiled file holds
    this text."""
    import sysconfig

    import torch

    return f"torch {torch.__version__}, {sysconfig.get_config_var('SOABI')}"


def _binding_stale(newest_src: float) -> bool:
    return (not BINDING_PATH.exists() or BINDING_PATH.stat().st_mtime < newest_src
            or built_for().encode() not in BINDING_PATH.read_bytes())


def _compile_binding() -> None:
    """csrc/binding.cpp (host code only) against the installed torch."""
    import sysconfig

    import torch

    root = Path(torch.__path__[0])
    inc = [root / "include", root / "include" / "torch" / "csrc" / "api" / "include", sysconfig.get_paths()["include"],
           Path(_hipcc()).resolve().parents[1] / "include"]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", f'-DLQ_BUILT_FOR="{built_for()}"', *(f"-I{i}" for i in inc), str(CSRC / "binding.cpp"),
           "-o", str(BINDING_PATH), f"-L{root / 'lib'}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on binding.cpp:\n{res.stderr}")


def _bind(force: bool, newest_src: float) -> None:
    if force or _binding_stale(newest_src):
        _compile_binding()


def build(force: bool = True, jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every .hip source and link the shared library, then report the native host code if that failed: the C library needs
    hipcc alone. Returns the library path."""
    srcs = sources()
    objdir = CSRC / "build"
    objdir.mkdir(exist_ok=True)
    headers = list(CSRC.glob("*.h")) + [CSRC.parents[1] / "include" / "linquant_hip.h"]
    newest_hdr = max(h.stat().st_mtime for h in headers)
    todo = []
    for s in srcs:
        o = objdir / (s.stem + ".o")
        if force or not o.exists() or o.stat().st_mtime < max(s.stat().st_mtime, newest_hdr):
            todo.append((s, o))
    jobs = jobs or min(8, max(1, (os.cpu_count() or 2)))
    if verbose:
        print(f"[linquant_amd.build] compiling {len(todo)}/{len(srcs)} sources with {jobs} jobs", flush=True)
    bind = CSRC / "binding.cpp"
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        binding = ex.submit(_bind, force, max(bind.stat().st_mtime, newest_hdr))
        list(ex.map(lambda so: _compile(*so), todo))
    objs = [str(objdir / (s.stem + ".o")) for s in srcs]
    cmd = [_hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", str(LIB_PATH)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    failure = binding.exception()
    if failure is not None:
        raise RuntimeError(f"{LIB_PATH.name} is built, the Python wrappers' {BINDING_PATH.name} is not: {failure}") from failure
    return LIB_PATH


if __name__ == "__main__":
    path = build(force="--incremental" not in sys.argv, verbose=True)
    print(path)
