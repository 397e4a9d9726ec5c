"""Build libdecodebench_hip.so in-tree with hipcc for gfx950.

    python -m decodebench_amd.build          # compile if sources changed
    python -m decodebench_amd.build --force  # always recompile

Every HIP source under ``csrc/`` is compiled to an object in ``_build/`` (in
parallel), then linked into ``decodebench_amd/lib/libdecodebench_hip.so``.
All device code is built with packed-fp32 instructions disabled
(``-Xclang -target-feature -Xclang -packed-fp32-ops``); the host pass warns
that it does not know that feature, which is expected.

``csrc/fastcall.cpp``, the native call path of the Python ops, is host code
built against the installed torch into ``lib/_fastcall.so`` where g++ and the
headers for it are there; the ops work without it.
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
import warnings
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
LIB_DIR = PKG / "lib"
LIB = LIB_DIR / "libdecodebench_hip.so"
FAST_SRC = CSRC / "fastcall.cpp"
FAST_LIB = LIB_DIR / "_fastcall.so"
INCLUDE = PKG.parent / "include"

ARCH = os.environ.get("DECODEBENCH_OFFLOAD_ARCH", "gfx950")
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
    f"-I{INCLUDE}", f"-I{CSRC}",
]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; the HIP toolchain is required to build")
    return path


def _sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


def _headers() -> list[Path]:
    return sorted(CSRC.glob("*.h")) + sorted(INCLUDE.glob("*.h"))


def _stale(obj: Path, src: Path) -> bool:
    if not obj.exists():
        return True
    newest = max([src.stat().st_mtime] + [h.stat().st_mtime for h in _headers()])
    return obj.stat().st_mtime < newest


def _compile(src: Path) -> Path:
    obj = BUILD / (src.stem + ".o")
    cmd = [hipcc(), *HIP_FLAGS, "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src.name}:\n{res.stderr}")
    return obj


def _fast_stale() -> bool:
    """Whether the native call path is missing, older than its sources or built
    for another torch or Python (which its file holds as a text)."""
    from decodebench_amd.ops import fast_built_for

    return _stale(FAST_LIB, FAST_SRC) or fast_built_for().encode() not in FAST_LIB.read_bytes()


def _compile_fast(src: Path) -> Path:
    import torch

    from decodebench_amd.ops import fast_built_for

    root = Path(torch.__file__).resolve().parent
    tmp = FAST_LIB.with_suffix(".so.tmp")
    abi = int(getattr(torch._C, "_GLIBCXX_USE_CXX11_ABI", True))
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-shared",
           f"-D_GLIBCXX_USE_CXX11_ABI={abi}", f'-DDB_BUILT_FOR="{fast_built_for()}"',
           f"-I{sysconfig.get_paths()['include']}",
           f"-I{root / 'include'}", f"-I{root / 'include/torch/csrc/api/include'}", str(src),
           "-o", str(tmp), f"-L{root / 'lib'}", "-ltorch_python", "-ltorch_cpu", "-lc10"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for {src.name}:\n{res.stderr}")
    os.replace(tmp, FAST_LIB)
    return FAST_LIB


def _build_fast(force: bool) -> None:
    """Build the native call path where that takes a build.  The ops work
    without it, so a host that cannot build it (no torch, no headers, no g++)
    gets a warning; a file that its sources have outgrown does not stay."""
    try:
        if force or _fast_stale():
            _compile_fast(FAST_SRC)
    except Exception as exc:
        FAST_LIB.unlink(missing_ok=True)
        warnings.warn(f"the native call path of the ops was not built: {exc}", stacklevel=2)


def build(force: bool = False, verbose: bool = True) -> Path:
    """Compile the HIP library and the native call path; return the path of
    the library."""
    BUILD.mkdir(exist_ok=True)
    LIB_DIR.mkdir(exist_ok=True)
    srcs = _sources()
    todo = [s for s in srcs if force or _stale(BUILD / (s.stem + ".o"), s)]
    workers = min(len(todo) + 1, max(1, (os.cpu_count() or 2)))
    with cf.ThreadPoolExecutor(max_workers=workers) as pool:
        fast = pool.submit(_build_fast, force)
        list(pool.map(_compile, todo))
        fast.result()
    objs = [BUILD / (s.stem + ".o") for s in srcs]
    if force or todo or not LIB.exists() or any(
            o.stat().st_mtime > LIB.stat().st_mtime for o in objs):
        tmp = LIB.with_suffix(".so.tmp")
        cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC",
               *map(str, objs), "-o", str(tmp)]
        res = subprocess.run(cmd, capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"link failed:\n{res.stderr}")
        os.replace(tmp, LIB)
    if verbose:
        print(f"[decodebench_amd.build] {LIB} ({len(todo)} of {len(srcs)} sources compiled)")
    return LIB


def main(argv=None) -> int:
    ap = argparse.ArgumentParser(description=__doc__.splitlines()[0])
    ap.add_argument("--force", action="store_true")
    args = ap.parse_args(argv)
    build(force=args.force)
    return 0


if __name__ == "__main__":
    sys.exit(main())
