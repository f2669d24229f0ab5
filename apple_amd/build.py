"""Build the HIP library ``apple_amd/_lib/libapple_amd.so`` for gfx950.

Each ``csrc/*.hip`` and ``csrc/*.cpp`` file is compiled with hipcc in
parallel and linked into one shared object with a C ABI (declared in
``include/apple_amd.h``).  Packed-FP32 instructions are disabled for all
device code.  ``csrc/python/tensor_calls.cpp`` becomes the extension module
``apple_amd/_lib/tensor_calls.so`` (host code against PyTorch's headers).
"""

from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "_lib")
OBJDIR = os.path.join(HERE, "_lib", "obj")
LIBNAME = "libapple_amd.so"
MODULE = "tensor_calls"
ARCH = os.environ.get("APPLE_AMD_ARCH", "gfx950")

DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
COMMON = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-result", "-Wno-unused-variable"]


def hipcc() -> str:
    path = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(path):
        raise RuntimeError("hipcc not found: the ROCm toolchain is required to build apple_amd")
    return path


def sources() -> list[str]:
    return sorted(
        os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp"))
    )


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, os.path.basename(src) + ".o")
    cmd = [hipcc(), *COMMON, "-c", src, "-o", obj]
    if src.endswith(".hip"):
        cmd[1:1] = ["-x", "hip", *DEVICE_FLAGS]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    return obj


def _build_module() -> None:
    """The extension module that calls the library from torch tensors."""
    import torch
    from torch.utils import cpp_extension

    out = os.path.join(LIBDIR, MODULE + ".so")
    include = [sysconfig.get_paths()["include"], *cpp_extension.include_paths()]
    cmd = [
        hipcc(), *COMMON, "-shared", os.path.join(CSRC, "python", MODULE + ".cpp"), "-o", out + ".tmp",
        *(f"-isystem{p}" for p in include), f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
        *(f"-L{p}" for p in cpp_extension.library_paths()), "-lc10", "-ltorch_cpu", "-ltorch_python",
    ]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
    os.replace(out + ".tmp", out)


def build(verbose: bool = True) -> str:
    """Compile every source and link the shared library, then the extension
    module (left out where there is no PyTorch: the C ABI needs none);
    returns the library's path."""
    os.makedirs(OBJDIR, exist_ok=True)
    srcs = sources()
    jobs = min(len(srcs) + 1, max(1, min(16, os.cpu_count() or 1)))
    with concurrent.futures.ThreadPoolExecutor(jobs) as ex:
        module = ex.submit(_build_module)
        objs = list(ex.map(_compile, srcs))
        out = os.path.join(LIBDIR, LIBNAME)
        tmp = out + ".tmp"
        cmd = [hipcc(), "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp]
        proc = subprocess.run(cmd, capture_output=True, text=True)
        if proc.returncode != 0:
            raise RuntimeError(f"link failed: {' '.join(cmd)}\n{proc.stdout}\n{proc.stderr}")
        os.replace(tmp, out)
        try:
            module.result()
        except ImportError as e:
            print(f"{MODULE}.so not built: {e}", file=sys.stderr)
    if verbose:
        print(f"built {out}", file=sys.stderr)
    return out


if __name__ == "__main__":
    build()
