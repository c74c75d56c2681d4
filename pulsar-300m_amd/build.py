"""Build libpulsar_hip.so (gfx950) from csrc/ with hipcc, and the op surface's native half
(_ops.so, host code against torch's headers), in place.

    python pulsar-300m_amd/build.py [--jobs N]

Objects are compiled in parallel into _build/ next to this file; the shared libraries are
written to pulsar_cuda/, where the pulsar_cuda package loads them.
"""

from __future__ import annotations

import argparse
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "pulsar_cuda", "libpulsar_hip.so")
OPS_OUT = os.path.join(HERE, "pulsar_cuda", "_ops.so")
BUILD = os.path.join(HERE, "_build")
SOURCES = ["ops.hip", "gemm.hip", "gemm_wide.hip", "gemm_f32.hip", "rows.hip", "sample.hip", "engine.hip", "backward.hip"]
ARCH = os.environ.get("PULSAR_HIP_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    # packed fp32 instructions are left to the compiler's scalar/float2 code only
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _compile(src: str) -> str:
    obj = os.path.join(BUILD, src.replace(".hip", ".o"))
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"hipcc failed on {src}")
    return obj


def _run(cmd: list, what: str) -> None:
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError(f"{what} failed")


def _compile_ops() -> str:
    """Host code of the op surface, against the headers of the installed torch."""
    import sysconfig

    import torch

    t = os.path.dirname(torch.__file__)
    obj = os.path.join(BUILD, "ops_torch.o")
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    _run([HIPCC, "-x", "c++", "-O2", "-std=c++17", "-fPIC", "-w", "-DUSE_ROCM=1",
          "-D__HIP_PLATFORM_AMD__=1", f"-D_GLIBCXX_USE_CXX11_ABI={abi}", f"-I{t}/include",
          f"-I{t}/include/torch/csrc/api/include", "-I" + sysconfig.get_path("include"),
          "-I" + os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"),
          "-c", os.path.join(CSRC, "ops_torch.cpp"), "-o", obj], "ops_torch.cpp")
    return obj


def _link_ops(obj: str) -> None:
    import torch

    t = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = OPS_OUT + ".tmp"
    _run([HIPCC, "-shared", "-fPIC", "-no-hip-rt", obj, "-o", tmp, f"-L{t}", "-lc10", "-lc10_hip",
          "-ltorch_cpu", "-ltorch_python", "-L" + os.path.dirname(OUT), "-l:libpulsar_hip.so",
          "-Wl,-rpath,$ORIGIN"], "link of _ops.so")
    os.replace(tmp, OPS_OUT)


def build(jobs: int = 8) -> str:
    os.makedirs(BUILD, exist_ok=True)
    with ThreadPoolExecutor(max(1, jobs)) as ex:
        ops = ex.submit(_compile_ops)
        objs = list(ex.map(_compile, SOURCES))
        ops_obj = ops.result()
    tmp = OUT + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp], "link")
    os.replace(tmp, OUT)
    _link_ops(ops_obj)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=min(8, os.cpu_count() or 1))
    print(build(ap.parse_args().jobs))
