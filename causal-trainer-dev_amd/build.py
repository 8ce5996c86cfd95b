"""Build recipe for libct_hotpath.so (HIP, gfx950 only) and _native.so (its torch side, host code).

Run ``python causal-trainer-dev_amd/build.py`` (or call :func:`build`) on any
machine with hipcc; no GPU is needed to compile. The libraries are placed
next to this file: libct_hotpath.so is what :mod:`_lib` loads through ctypes and what
_native.so links, _native.so the extension module the torch operators call. The first needs
nothing but hipcc; the second also g++ and torch, and is left out where torch is not installed.
"""

from __future__ import annotations

import importlib.util
import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
CSRC = PACKAGE_DIR / "csrc"
LIBRARY = PACKAGE_DIR / "libct_hotpath.so"
NATIVE = PACKAGE_DIR / "_native.so"
SOURCES = ("ct_error.hip", "ct_attn.hip", "ct_cutce.hip", "ct_prep.hip", "ct_layer.hip", "ct_logits_ce.hip")

# -packed-fp32-ops is switched off on purpose: hipcc must not form packed FP32
# instructions from scalar float code on this target.
HIP_FLAGS = (
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-value",
    "-Wno-inline-asm",
)


def hipcc() -> str:
    found = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(found):
        raise RuntimeError("hipcc not found; libct_hotpath.so needs the ROCm toolchain")
    return found


def _run(cmd: list[str]) -> None:
    result = subprocess.run(cmd, capture_output=True, text=True)
    if result.returncode != 0:
        sys.stderr.write(result.stdout + result.stderr)
        raise RuntimeError("command failed: " + " ".join(cmd))


def build(verbose: bool = False, extra_flags: tuple[str, ...] = ()) -> Path:
    """Compile every HIP source and link libct_hotpath.so, then _native.so. Always recompiles."""

    compiler = hipcc()
    build_dir = PACKAGE_DIR / "build"
    build_dir.mkdir(exist_ok=True)
    sources = [name for name in SOURCES if (CSRC / name).exists()]
    objects = [build_dir / (Path(name).stem + ".o") for name in sources]

    def compile_one(pair):
        name, obj = pair
        cmd = [compiler, *HIP_FLAGS, *extra_flags, "-c", str(CSRC / name), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    native_object = build_dir / "ct_torch.o"
    with_torch = importlib.util.find_spec("torch") is not None
    with ThreadPoolExecutor(max_workers=4) as pool:
        native = pool.submit(_compile_native, native_object, verbose) if with_torch else None
        list(pool.map(compile_one, zip(sources, objects)))
    link = [compiler, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", "-Wl,-soname,libct_hotpath.so",
            *map(str, objects), "-o", str(LIBRARY)]
    if verbose:
        print(" ".join(link), flush=True)
    _run(link)
    if native is None:
        print(f"torch is not installed: {NATIVE.name}, which the torch operators need, is not built", file=sys.stderr)
        return LIBRARY
    native.result()
    _link_native(native_object, verbose)
    return LIBRARY


def _torch_paths():
    import torch

    root = Path(torch.__file__).resolve().parent
    return root / "include", root / "lib"


def _compile_native(obj: Path, verbose: bool) -> None:
    import sysconfig

    include, _ = _torch_paths()
    cmd = ["g++", "-c", str(CSRC / "ct_torch.cc"), "-o", str(obj), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden",
           "-DTORCH_EXTENSION_NAME=_native", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-Wno-attributes",
           f"-I{include}", f"-I{include / 'torch/csrc/api/include'}", "-I/opt/rocm/include",
           f"-I{sysconfig.get_paths()['include']}"]
    if verbose:
        print(" ".join(cmd), flush=True)
    _run(cmd)


def _link_native(obj: Path, verbose: bool) -> None:
    _, lib = _torch_paths()
    cmd = ["g++", "-shared", str(obj), "-o", str(NATIVE), str(LIBRARY), "-Wl,-rpath,$ORIGIN", f"-L{lib}",
           f"-Wl,-rpath,{lib}", "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch", "-ltorch_python"]
    if verbose:
        print(" ".join(cmd), flush=True)
    _run(cmd)


if __name__ == "__main__":
    print(build(verbose=True))
