"""Builds libpllm_hip.so (gfx950) in-tree with hipcc.

    python -m pocketllm_amd.build

One object per csrc/*.hip, compiled in parallel, linked into pocketllm_amd/libpllm_hip.so; then the native host path of the Python
operators (csrc/bindings.cpp, against this library and the installed torch) into pocketllm_amd/_bindings.so.
"""
from __future__ import annotations

import concurrent.futures
import importlib.util
import os
import subprocess
import sys
import sysconfig
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
OBJ_DIR = PKG / "build"
LIB = PKG / "libpllm_hip.so"
BINDINGS = PKG / "_bindings.so"

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-inline-asm",
]


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in proc.stdout.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"command failed ({proc.returncode}): {' '.join(cmd)}\n{out}")
    if out.strip():
        print(out, file=sys.stderr)


def _build_bindings() -> None:
    """csrc/bindings.cpp: host code only, so the host compiler; torch's libraries are in the process before it is imported."""
    torch_dir = Path(importlib.util.find_spec("torch").origin).parent
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    _run(["g++", "-std=c++17", "-O2", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-I{torch_dir / 'include'}", f"-I{rocm}/include",
          f"-I{sysconfig.get_paths()['include']}", str(CSRC / "bindings.cpp"), "-o", str(BINDINGS), f"-L{torch_dir / 'lib'}", "-ltorch_python",
          "-ltorch_cpu", "-lc10", "-lc10_hip", f"-L{PKG}", "-lpllm_hip", "-Wl,-rpath,$ORIGIN"])


def build_library(verbose: bool = True, jobs: int = 8, incremental: bool = False) -> Path:
    """Compiles every csrc/*.hip and links the library.  incremental=True (python -m pocketllm_amd.build --incremental) skips
    sources whose object file is newer than the source and than every header."""
    OBJ_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    objs = [OBJ_DIR / (s.stem + ".o") for s in sources]
    newest_header = max(h.stat().st_mtime for h in [*CSRC.glob("*.h"), *CSRC.glob("*.inc"), *(PKG.parent / "include").glob("*.h")])
    todo = [(s, o) for s, o in zip(sources, objs)
            if not (incremental and o.exists() and o.stat().st_mtime > max(s.stat().st_mtime, newest_header))]
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as pool:
        futs = [pool.submit(_run, ["hipcc", *HIPCC_FLAGS, "-c", str(s), "-o", str(o)]) for s, o in todo]
        for f in futs:
            f.result()
    _run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *map(str, objs), "-o", str(LIB)])
    _build_bindings()
    if verbose:
        print(f"built {LIB} from {len(sources)} sources")
    return LIB


if __name__ == "__main__":
    build_library(incremental="--incremental" in sys.argv[1:])
