"""Builds libmoe_hip.so (the C-ABI library of HIP kernels) for gfx950 with hipcc and, where torch is there, the extension
moe_call.

Run on the CPU host: hipcc cross-compiles without a GPU.  The library is written
next to this file so that it travels with the source tree.
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB_PATH = os.path.join(HERE, "libmoe_hip.so")
# the timing probe of the grouped GEMM's K loop (`python bench.py --probe`): its own library, nothing of the product links it
PROBE_PATH = os.path.join(HERE, "libmoe_probe.so")

# the layer calls' host work (a Python extension over torch's headers; it gets the library's functions by address).  The suffix is the
# interpreter's: another one does not find it.
CALL_PATH = os.path.join(HERE, "moe_call" + sysconfig.get_config_var("EXT_SUFFIX"))

SOURCES = ["moe_api.hip", "moe_route.hip", "moe_router.hip", "moe_permute.hip", "moe_quant.hip", "moe_gemm.hip", "moe_gemm_stream.hip",
           "moe_token.hip", "moe_small.hip", "moe_combine.hip"]
# no v_pk_*_f32 code generation (some packed-f32 forms have given wrong results on this hardware)
COMMON = ["--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function",
          "-fvisibility=hidden",    # only the functions include/moe_hip.h declares (MOE_API) are exported
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-I", os.path.join(ROOT, "include"), "-I", CSRC]
# routing (also of single tokens, moe_token.hip) and combine promise individually rounded f32 operations (bit-reproducible on a CPU)
PER_FILE = {"moe_route.hip": ["-ffp-contract=off"], "moe_combine.hip": ["-ffp-contract=off"],
            "moe_router.hip": ["-ffp-contract=off", "-Wno-inline-asm"],
            # MFMA results go straight to VGPRs: the block-scale FMA consumes them on the vector ALU
            "moe_gemm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-Wno-inline-asm"],   # m0 is clobbered on purpose
            "moe_gemm_stream.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-Wno-inline-asm"],
            "moe_token.hip": ["-ffp-contract=off", "-mllvm", "-amdgpu-mfma-vgpr-form", "-Wno-inline-asm"],
            "moe_small.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form", "-Wno-inline-asm"]}


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: the MI355X kernels cannot be built")


def _call_command() -> list[str] | None:
    """None without torch, which nothing but the extension needs."""
    try:
        import torch
    except ImportError:
        return None
    base = os.path.dirname(torch.__file__)
    return [shutil.which("g++") or "g++", "-O2", "-shared", "-fPIC", "-std=c++17", "-Wall", "-fvisibility=hidden",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}", "-I", os.path.join(ROOT, "include"),
            "-isystem", os.path.join(base, "include"), "-isystem", sysconfig.get_paths()["include"],
            os.path.join(CSRC, "moe_call.cpp"), "-o", CALL_PATH, "-L", os.path.join(base, "lib"), "-lc10", "-ltorch_cpu", "-ltorch_python"]


def build(verbose: bool = True, jobs: int = 6) -> str:
    hipcc = _hipcc()
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [hipcc, *COMMON, *PER_FILE.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
        if len(procs) >= jobs:
            _drain(procs)
    _drain(procs)
    probe = [hipcc, *COMMON, *PER_FILE["moe_gemm.hip"], "-shared", os.path.join(CSRC, "moe_probe.hip"), "-o", PROBE_PATH]
    if verbose:
        print(" ".join(probe), flush=True)
    procs.append(("moe_probe.hip", subprocess.Popen(probe, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB_PATH]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)
    # (last: whatever becomes of the extension, the library is there)
    call = _call_command()
    if call is None:
        print("moe_call.cpp is left out: it needs torch", flush=True)
    else:
        if verbose:
            print(" ".join(call), flush=True)
        procs.append(("moe_call.cpp", subprocess.Popen(call, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    _drain(procs)
    return LIB_PATH


def _drain(procs):
    while procs:
        src, p = procs.pop(0)
        out, _ = p.communicate()
        out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip())
        if out:
            print(out, flush=True)
        if p.returncode != 0:
            raise RuntimeError(f"the compiler failed on {src}")


if __name__ == "__main__":
    print(build(verbose="-q" not in sys.argv))
