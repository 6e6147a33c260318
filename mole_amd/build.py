"""Builds MOLE/cpp/libmole_hip.so (gfx950 only) with hipcc, from the sources beside it: the native extension sits
where the reference keeps its own (MOLE/cpp); and mole_torch.so, the layer's autograd node on top of its C ABI (host code
against torch's headers).  `python -m mole_amd.build`."""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CPP = os.path.join(ROOT, "MOLE", "cpp")
LIB = os.path.join(CPP, "libmole_hip.so")
SOURCES = ["error.cpp", "route.hip", "permute.hip", "ffn_gemm.hip", "gemm256.hip", "gemm_f32.hip", "gemm_skinny.hip", "layer.hip", "adam.hip", "unimem.hip", "probe.hip"]
TORCH_LIB = os.path.join(CPP, "mole_torch.so")
TORCH_SOURCE = "torch_layer.cpp"
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-x", "hip",
         # keep the compiler from forming packed-fp32 VALU ops
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument",
         "-I" + os.path.join(ROOT, "include"), "-I" + CPP]
# MOLE_TUNING=1 in the environment of the build adds the launch orders and K-loop ablations that were measured against
# the defaults (selected at run time by MOLE_MFAST, MOLE_GEMM, ...: see MOLE/cpp/gemm256.hip and ffn_gemm.hip)
if os.environ.get("MOLE_TUNING"):
    FLAGS.append("-DMOLE_TUNING")


def _compile(src: str) -> str:
    obj = os.path.join(CPP, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CPP, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines()
                     if "packed-fp32-ops" not in l and l.strip())
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{msgs}")
    if msgs:
        print(msgs, file=sys.stderr)
    return obj


def _run(cmd, what):
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{what} failed:\n" + r.stdout + r.stderr)


def _compile_torch() -> str:
    import torch
    from torch.utils.cpp_extension import include_paths
    obj = os.path.join(CPP, "torch_layer.o")
    flags = ["-O2", "-std=c++17", "-fPIC", "-w", "-DTORCH_EXTENSION_NAME=mole_torch", "-DTORCH_API_INCLUDE_EXTENSION_H",
             f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM",
             "-I" + os.path.join(ROOT, "include"), "-I" + sysconfig.get_paths()["include"]]
    flags += [f for p in include_paths("cuda") for f in ("-isystem", p)]
    _run([HIPCC, *flags, "-c", os.path.join(CPP, TORCH_SOURCE), "-o", obj], "hipcc on " + TORCH_SOURCE)
    return obj


def _link_torch(obj: str) -> None:
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run([HIPCC, "-shared", "-fPIC", "-o", TORCH_LIB, obj, "-L" + CPP, "-l:libmole_hip.so", "-Wl,-rpath,$ORIGIN", "-L" + lib,
          "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"], "link of mole_torch.so")


def build(verbose: bool = False) -> str:
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CPP, s))]
    missing = sorted(set(SOURCES) - set(srcs))
    if missing:
        raise RuntimeError(f"missing sources: {missing}")
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        torch_obj = ex.submit(_compile_torch)         # the longest of the compilations
        objs = list(ex.map(_compile, srcs))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    _link_torch(torch_obj.result())
    if verbose:
        print("built", LIB, TORCH_LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True)
