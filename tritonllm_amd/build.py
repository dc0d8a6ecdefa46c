"""Compile the HIP sources into ``tritonllm_amd/lib/libtllm_hip.so`` for gfx950, and the host side of the ops next to it.

``hipcc`` cross-compiles without a GPU, so this runs anywhere the ROCm toolchain
is installed. Usage: ``python -m tritonllm_amd.build``.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libtllm_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "tllm_host.so")
INCLUDE = os.path.join(ROOT, "include")

SOURCES = ["abi.hip", "rmsnorm.hip", "embedding.hip", "swiglu.hip", "rope.hip", "qkv_decode.hip", "qkv_decode_r8.hip", "qkv_decode_r32.hip", "qkv_decode_rows.hip", "qkv_prefill.hip", "tile_gemm.hip", "decode_general.hip", "out_decode.hip", "out_decode_r8.hip", "out_decode_r32.hip", "unembed.hip", "unembed_tiles.hip", "attn_decode.hip", "attn_prefill.hip", "mxfp4.hip"]

# -packed-fp32-ops: keep the compiler from forming v_pk_*_f32 from ordinary float code.
HIPCC_FLAGS = [
    "-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
] + os.environ.get("TLLM_EXTRA_HIPCC_FLAGS", "").split()


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found: the ROCm toolchain is required to build libtllm_hip.so")
    return exe


def _compile(src: str, obj_dir: str) -> str:
    obj = os.path.join(obj_dir, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, "-I", INCLUDE, "-I", CSRC, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stdout}\n{r.stderr}")
    return obj


def _compile_host(out: str) -> None:
    """The Python-side half (csrc/host_ops.cpp): plain C++ against torch's headers, linked to the kernels' library."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths

    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(_hipcc())))
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE, *(f"-I{d}" for d in include_paths()),
           f"-I{os.path.join(rocm, 'include')}", f"-I{sysconfig.get_paths()['include']}", os.path.join(CSRC, "host_ops.cpp"), "-o", out,
           f"-L{LIB_DIR}", "-ltllm_hip", f"-L{torch_lib}", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed on host_ops.cpp:\n{r.stdout}\n{r.stderr}")


def build_library(verbose: bool = False) -> str:
    obj_dir = os.path.join(PKG_DIR, "build")
    os.makedirs(obj_dir, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(lambda s: _compile(s, obj_dir), SOURCES))
    tmp = LIB_PATH + ".tmp"
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    _compile_host(HOST_PATH + ".tmp")
    os.replace(HOST_PATH + ".tmp", HOST_PATH)
    if verbose:
        for p in (LIB_PATH, HOST_PATH):
            print(f"built {p} ({os.path.getsize(p)} bytes)")
    return LIB_PATH


if __name__ == "__main__":
    build_library(verbose=True)
    sys.exit(0)
