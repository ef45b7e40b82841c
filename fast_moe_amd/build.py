"""Builds libfastmoe_hip.so (gfx950) from fast_moe_amd/csrc with hipcc, in-tree.

    python -m fast_moe_amd.build            # compile every translation unit and link
    python -m fast_moe_amd.build --out fast_moe_amd/libfastmoe_hip_trace.so -DFMOE_TRACE
                                            # a second library beside it (here: the debug build whose
                                            # ring kernel records per-tile time stamps; load it with
                                            # FMOE_LIB_PATH=<that file>, see bench.py --tile-trace)
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_PATH = os.path.join(HERE, "libfastmoe_hip.so")
HOST_PATH = os.path.join(HERE, "_host.so")     # the native side of the Python wrappers (csrc/host_calls.cpp)
OBJ_DIR = os.path.join(CSRC, "build")

SOURCES = ["gemm_bf16.hip", "gemm_fp8.hip", "gemm_bf16_tail.hip", "gemm_fp8_tail.hip", "gemm_bf16_short.hip", "gemm_fp8_short.hip",
           "gemm_bf16_split.hip", "gemm_fp8_split.hip", "gemm_f32.hip", "gemm_direct.hip", "gemm_wgrad.hip", "gemm_api.hip",
           "gate.hip", "core.hip", "routing.hip", "quant.hip", "combine.hip", "backward.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    # keep the compiler from forming packed fp32 VALU ops out of scalar float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _compile(src: str, extra, obj_dir: str = OBJ_DIR) -> str:
    obj = os.path.join(obj_dir, os.path.splitext(src)[0] + ".o")
    cmd = [_hipcc(), *HIPCC_FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    return obj


def _build_host() -> str:
    """The extension module that issues the forward operators' calls: plain C++ against torch's headers."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *(f"-isystem{p}" for p in cpp_extension.include_paths()), "-isystem" + sysconfig.get_paths()["include"],
           os.path.join(CSRC, "host_calls.cpp"), "-o", HOST_PATH, "-L" + torch_lib,
           "-ltorch_cpu", "-ltorch", "-lc10", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for host_calls.cpp:\n{res.stdout}\n{res.stderr}")
    return HOST_PATH


def build(extra_flags=(), jobs: int = 8, verbose: bool = True, out: str = LIB_PATH) -> str:
    # (a library under another name keeps its objects apart from the product's)
    obj_dir = OBJ_DIR if os.path.abspath(out) == LIB_PATH else os.path.join(OBJ_DIR, os.path.splitext(os.path.basename(out))[0])
    os.makedirs(obj_dir, exist_ok=True)
    with ThreadPoolExecutor(max_workers=max(1, min(jobs, len(SOURCES)))) as pool:
        # (a library under another name goes with the product's extension module, which takes its entry points by address)
        host = pool.submit(_build_host) if obj_dir == OBJ_DIR else None
        objs = list(pool.map(lambda s: _compile(s, list(extra_flags), obj_dir), SOURCES))
    if host is not None:
        host.result()
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *objs]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    if verbose:
        print(f"built {out} ({os.path.getsize(out) / 1e6:.1f} MB)")
    return out


if __name__ == "__main__":
    args = sys.argv[1:]
    target = LIB_PATH
    if "--out" in args:
        i = args.index("--out")
        target = os.path.abspath(args[i + 1])
        del args[i:i + 2]
    build(extra_flags=args, out=target)
