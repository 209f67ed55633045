"""Builds libmoe_i8.so (HIP kernels + C-ABI) for gfx950 with hipcc, in-tree, and, as a step of its own, the native
call path of the Python entry points (_host.so), which needs g++ and the installed torch's headers."""

from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
LIB_PATH = PKG_DIR / "libmoe_i8.so"
SOURCES = ["align.hip", "quant.hip", "sum.hip", "router.hip", "gemm_stream.hip", "gemm_tile.hip", "gemm_wide.hip",
           "gemm_deep.hip", "gemm_narrow.hip", "gemm_dense.hip", "gemm_dense_rows.hip", "gemm_split.hip", "few_tokens.hip", "dense_few.hip", "api.hip"]
HOST_PATH = PKG_DIR / "_host.so"  # the Python entry points' native call path (CPython extension, no device code)
PROBE_LIB_PATH = PKG_DIR / "libmoe_i8_probe.so"  # the benchmark's MFMA rate probe, a library of its own

# packed-fp32 VALU ops are switched off for all device code (hipcc's host pass warns that it does
# not know the feature; that is harmless).
HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Wno-inline-asm",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _run(cmd: list[str]) -> None:
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError("command failed: " + " ".join(cmd) + "\n" + proc.stdout + proc.stderr)


def build_library(verbose: bool = False) -> Path:
    """Compile every HIP source to an object file and link libmoe_i8.so and the benchmark's probe library. Needs hipcc
    only. Always rebuilds."""
    hipcc = _hipcc()
    objdir = PKG_DIR / "build"
    objdir.mkdir(exist_ok=True)
    objs = [objdir / (Path(s).stem + ".o") for s in SOURCES]
    probe_obj = objdir / "probe.o"

    def compile_one(pair):
        src, obj = pair
        cmd = [hipcc, *HIPCC_FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        _run(cmd)

    with ThreadPoolExecutor(max_workers=8) as pool:
        list(pool.map(compile_one, zip([*SOURCES, "probe.hip"], [*objs, probe_obj])))
    for path, parts in ((LIB_PATH, objs), (PROBE_LIB_PATH, [probe_obj])):
        tmp = path.with_suffix(".so.tmp")
        _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *map(str, parts), "-o", str(tmp)])
        os.replace(tmp, path)
    return LIB_PATH


def build_host() -> Path:
    """Compile the CPython extension against the installed torch and link it with libmoe_i8.so, which is there already.
    Host code only. Without it the Python entry points make the same calls through ctypes."""
    import torch

    lib = Path(torch.__path__[0])
    objdir = PKG_DIR / "build"
    objdir.mkdir(exist_ok=True)
    obj, tmp = objdir / "host.o", HOST_PATH.with_suffix(".so.tmp")
    includes = [lib / "include", lib / "include/torch/csrc/api/include", "/opt/rocm/include", sysconfig.get_paths()["include"]]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", f'-DMOE_I8_TORCH_VERSION="{torch.__version__}"',
          *(arg for i in includes for arg in ("-isystem", str(i))), "-c", str(CSRC / "host.cpp"), "-o", str(obj)])
    _run(["g++", "-shared", str(obj), "-o", str(tmp), f"-L{PKG_DIR}", f"-l:{LIB_PATH.name}", "-Wl,-rpath,$ORIGIN",
          f"-L{lib / 'lib'}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-L/opt/rocm/lib", "-lamdhip64"])
    os.replace(tmp, HOST_PATH)
    return HOST_PATH


if __name__ == "__main__":
    print(build_library(verbose="-v" in sys.argv))
    print(build_host())
