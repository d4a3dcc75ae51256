"""Build recipe for libflagattention_amd.so (gfx950 only).

Compiles every HIP source under ``csrc/`` with hipcc for ``--offload-arch=gfx950``
and links them into ``flagattention_amd/libflagattention_amd.so`` in-tree, and the host
module ``flagattention_amd/_native.so`` (g++, against torch's headers) beside it, so that both
travel with the source tree.  Run ``python -m flagattention_amd.build``.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC_DIR = os.path.join(PKG_DIR, "csrc")
INCLUDE_DIR = os.path.join(REPO_DIR, "include")
BUILD_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "libflagattention_amd.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
NATIVE_SRC = os.path.join(CSRC_DIR, "host", "fa_native.cpp")
NATIVE_PATH = os.path.join(PKG_DIR, "_native.so")

ROCM_DIR = os.environ.get("ROCM_PATH", "/opt/rocm")
ARCH = "gfx950"
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # no packed fp32 VALU instructions (v_pk_*_f32) in any device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    f"-I{INCLUDE_DIR}",
    f"-I{CSRC_DIR}",
]
# Flags of single sources.  fa_decode_few.hip: MFMA accumulators in VGPRs.  Its LDS use allows
# one wave per SIMD, so the compiler would put them in AGPRs and copy them to and fro for the
# softmax rescale of every tile (32 rows: 122 us a step against 105).
SOURCE_FLAGS = {"fa_decode_few.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form=1"]}


def _hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found; ROCm is required to build flagattention_amd")
    return path


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC_DIR, f) for f in os.listdir(CSRC_DIR) if f.endswith(".hip")
    )


def native_object(verbose: bool = False) -> str:
    """Compile the host module (csrc/host/fa_native.cpp, against torch's headers)."""
    import torch

    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    obj = os.path.join(BUILD_DIR, "fa_native.o")
    cmd = [shutil.which("g++") or "g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f"-I{INCLUDE_DIR}", f"-I{inc}", f"-I{os.path.join(inc, 'torch/csrc/api/include')}",
           f"-I{ROCM_DIR}/include", f"-I{sysconfig.get_paths()['include']}",
           "-c", NATIVE_SRC, "-o", obj]
    _run(cmd, NATIVE_SRC, verbose)
    return obj


def link_native(obj: str, verbose: bool = False) -> None:
    """Link the host module against the library beside it and torch's libraries (which the
    importing process has loaded)."""
    import torch

    tmp = NATIVE_PATH + ".tmp"
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run([shutil.which("g++") or "g++", "-shared", obj, "-o", tmp, f"-L{PKG_DIR}",
          f"-l:{LIB_NAME}", f"-L{lib}", "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip",
          "-Wl,-rpath,$ORIGIN"], NATIVE_PATH, verbose)
    os.replace(tmp, NATIVE_PATH)


def _run(cmd: list[str], what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed for {what}:\n{res.stdout}\n{res.stderr}")


def build(verbose: bool = False) -> str:
    """Compile all HIP sources into the shared library and the host module beside it; returns
    the library's path."""
    hipcc = _hipcc()
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()

    def compile_one(src: str) -> str:
        obj = os.path.join(BUILD_DIR, os.path.basename(src)[:-4] + ".o")
        cmd = [hipcc, *HIPCC_FLAGS, *SOURCE_FLAGS.get(os.path.basename(src), []), "-c", src,
               "-o", obj]
        _run(cmd, src, verbose)
        return obj

    with concurrent.futures.ThreadPoolExecutor(max_workers=8) as ex:
        native = ex.submit(native_object, verbose)
        objs = list(ex.map(compile_one, srcs))
        native_obj = native.result()

    tmp = LIB_PATH + ".tmp"
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    _run(cmd, LIB_PATH, verbose)
    os.replace(tmp, LIB_PATH)
    link_native(native_obj, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
