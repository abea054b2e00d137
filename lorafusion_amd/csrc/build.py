"""Build liblorafusion_hip.so for gfx950 with hipcc (cross-compiles without a GPU), and the host module on top of it.

Usage: python -m lorafusion_amd.csrc.build   (or call build())
"""

from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB = os.path.join(PKG, "liblorafusion_hip.so")
HOST = os.path.join(PKG, "_host.so")
SOURCES = ["gemm_lora.hip", "gemm_big.hip", "gemm_mid.hip", "lora_skinny.hip", "lora_da_direct.hip", "lora_stream.hip", "nf4_dequant.hip", "dropout_mask.hip", "norm_act.hip", "lf_api.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++20", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-inline-asm",
]


# sources whose kernels issue memory instructions from inline assembly: their generated code is checked for the
# hazards the compiler does not resolve there (asm_lint.py)
LINTED = ["gemm_big.hip", "gemm_mid.hip", "gemm_lora.hip", "lora_skinny.hip", "lora_da_direct.hip", "lora_stream.hip"]


def _assembly(src: str) -> str:
    out = os.path.join(HERE, "build", src.replace(".hip", ".s"))
    cmd = ["hipcc", *FLAGS, "-S", "--cuda-device-only", os.path.join(HERE, src), "-o", out]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc -S failed on {src}:\n{res.stderr}")
    return out


def _compile(src: str) -> str:
    obj = os.path.join(HERE, "build", src.replace(".hip", ".o"))
    cmd = ["hipcc", *FLAGS, "-c", os.path.join(HERE, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_host() -> str:
    """host_ops.cpp (allocation, launches and autograd nodes: no GPU code) against torch's C++ headers."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(HERE, "build", "host_ops.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *[f"-I{i}" for i in cpp_extension.include_paths()],
           "-I/opt/rocm/include", f"-I{sysconfig.get_paths()['include']}", "-c", os.path.join(HERE, "host_ops.cpp"), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed on host_ops.cpp:\n{res.stderr}")
    return obj


def _link_host(obj: str) -> None:
    from torch.utils import cpp_extension

    cmd = ["g++", "-shared", "-fPIC", "-o", HOST, obj, *[f"-L{d}" for d in cpp_extension.library_paths()], "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_hip", "-ltorch", "-ltorch_python", f"-L{PKG}", "-llorafusion_hip", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link of the host module failed:\n{res.stderr}")


def build(verbose: bool = True) -> str:
    os.makedirs(os.path.join(HERE, "build"), exist_ok=True)
    from lorafusion_amd.csrc.asm_lint import lint

    with ThreadPoolExecutor(max_workers=6) as ex:
        host = ex.submit(_compile_host)
        asm = [ex.submit(_assembly, s) for s in LINTED]
        objs = list(ex.map(_compile, SOURCES))
        hazards = [v for a in asm for v in lint(a.result())]
    if hazards:
        raise RuntimeError("hazards in generated code that inline assembly hides from the compiler:\n" + "\n".join(hazards))
    res = subprocess.run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,-z,defs", "-o", LIB, *objs],
                         capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stderr}")
    _link_host(host.result())
    if verbose:
        print(f"built {LIB} and {HOST}")
    return LIB


if __name__ == "__main__":
    build()
