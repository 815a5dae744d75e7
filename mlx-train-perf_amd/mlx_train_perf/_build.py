"""Build the HIP C-ABI library in-tree for gfx950: ``python -m mlx_train_perf._build``.

Each HIP translation unit under ``csrc/`` is compiled by hipcc in parallel, then linked into
``mlx_train_perf/libmtp_hip.so`` next to this file (where ``_native`` loads it from). The autograd
nodes (``csrc/torch_nodes.cpp``, host code on torch's headers) become the extension module
``mlx_train_perf/_mtp_torch.so``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR.parent / "csrc"
OUT = PKG_DIR / "libmtp_hip.so"
NODE_SRC = CSRC / "torch_nodes.cpp"
NODE_OUT = PKG_DIR / "_mtp_torch.so"
OBJ_DIR = PKG_DIR.parent / "_build"
SOURCES = ("capi.hip", "lce_kernels.hip", "attn_kernels.hip", "f32_kernels.hip", "bench_probe.hip")
ARCH = os.environ.get("MTP_OFFLOAD_ARCH", "gfx950")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 arithmetic stays off: hipcc must not form v_pk_{add,mul,fma}_f32.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
]


def hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not Path(exe).exists():
        raise RuntimeError("hipcc not found (ROCm toolchain required to build the HIP extension)")
    return exe


def _compile(src: str) -> Path:
    obj = OBJ_DIR / (Path(src).stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", str(CSRC / src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stderr}")
    return obj


def _build_nodes() -> None:
    import torch

    root = Path(torch.__file__).resolve().parent
    rocm = Path(hipcc()).resolve().parents[1]
    tmp = NODE_OUT.with_suffix(".so.tmp")
    includes = [root / "include", root / "include/torch/csrc/api/include", rocm / "include", Path("/opt/rocm/include"),
                Path(sysconfig.get_paths()["include"])]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-isystem{p}" for p in includes), str(NODE_SRC), "-o", str(tmp), f"-L{root / 'lib'}", "-ltorch_python",
           "-ltorch_cpu", "-lc10", "-lc10_hip"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"compiling {NODE_SRC.name} failed:\n{res.stderr}")
    os.replace(tmp, NODE_OUT)


def build(verbose: bool = False) -> Path:
    OBJ_DIR.mkdir(exist_ok=True)
    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as ex:
        nodes = ex.submit(_build_nodes)
        objs = list(ex.map(_compile, SOURCES))
    tmp = OUT.with_suffix(".so.tmp")
    # --no-undefined: a kernel whose host launch stub was not emitted fails here, not at load time.
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,--no-undefined", "-o", str(tmp), *map(str, objs)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    os.replace(tmp, OUT)
    nodes.result()   # raises with the library in place: it serves every call without them
    if verbose:
        print(f"built {OUT} and {NODE_OUT.name}")
    return OUT


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
