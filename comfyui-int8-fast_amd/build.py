"""Build libi8f_gfx950.so from csrc/*.hip with hipcc and the host extension (_i8f_host.*.so) with g++, in-tree.

    python comfyui-int8-fast_amd/build.py [--force] [--keep-temps]

hipcc cross-compiles for gfx950 without a GPU.  The library is written next to
this file so that it travels with the source tree; nothing is installed.
"""
from __future__ import annotations

import argparse
import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
LIB = os.path.join(HERE, "libi8f_gfx950.so")
HOST_SRC = os.path.join(CSRC, "host", "i8f_host.cpp")

# -ffp-contract=off and correctly rounded division are part of the numerical
# contract (bit-exact quantiser, epilogue and merge); packed FP32 instructions
# are switched off for the device pass (the host pass does not know the feature
# and says so, harmlessly).
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-fast-math",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-kernarg-preload-count=16",
    "-DI8F_BUILD_CONTRACT=1",   # i8f_common.hpp refuses to compile without it: a build that bypasses these flags fails
    "-Wall",
    "-Wno-unused-function",
    "-Wno-inline-asm",   # the global->LDS loads name m0 in their clobber list, which clang reports as "reserved"
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; install ROCm or set HIPCC")


# gemm_i8_tiles.hip is compiled once per tile configuration and output type (names of csrc/gemm_i8_impl.hpp)
GEMM_CFGS = ("CfgBig", "CfgB192", "CfgTall", "CfgWide", "CfgMid", "CfgW96", "CfgMidDeep", "CfgM96Deep", "CfgS64Deep", "CfgT64Deep")
GEMM_GROUPED = ("CfgBig", "CfgB192", "CfgTall", "CfgWide")
GEMM_OUTS = ("OUT_BF16", "OUT_F16", "OUT_F32", "OUT_I32")


def units() -> list[tuple[str, str, list[str]]]:
    """(source, name of the object file, extra flags) of every compilation, the longest first."""
    out = []
    tiles = os.path.join(CSRC, "gemm_i8_tiles.hip")
    for cfg in GEMM_CFGS:
        for o in GEMM_OUTS:
            grouped = int(cfg in GEMM_GROUPED and o != "OUT_I32")
            out.append((tiles, f"gemm_i8_tiles_{cfg}_{o}.o", [f"-DI8F_TU_CFG={cfg}", f"-DI8F_TU_OUT={o}", f"-DI8F_TU_GROUPED={grouped}"]))
    for src in sorted(glob.glob(os.path.join(CSRC, "*.hip"))):
        if src != tiles:
            out.append((src, os.path.basename(src)[:-4] + ".o", []))
    return out


def _stale(target: str, deps: list[str]) -> bool:
    if not os.path.exists(target):
        return True
    t = os.path.getmtime(target)
    return any(os.path.getmtime(d) > t for d in deps)


def host_lib() -> str:
    """The host extension's file.  It is compiled against the layout of one torch's tensors and one Python's objects, so both
    are in its name: after an upgrade it is not found (and built again) instead of loaded."""
    import torch

    return os.path.join(HERE, f"_i8f_host.torch-{torch.__version__}.{sysconfig.get_config_var('SOABI')}.so")


def host_command() -> list[str]:
    """The compilation of the host extension (no device code: a CPython module against the installed torch)."""
    import torch

    t = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(hipcc())))
    include = [os.path.join(t, "include"), os.path.join(t, "include", "torch", "csrc", "api", "include"), sysconfig.get_paths()["include"],
               os.path.join(rocm, "include")]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            *(f for d in include for f in ("-isystem", d)), HOST_SRC, "-o", host_lib(), "-L" + os.path.join(t, "lib"),
            "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-Wl,-rpath," + os.path.join(t, "lib")]


def build(force: bool = False, keep_temps: bool = False, verbose: bool = True) -> str:
    cc = hipcc()
    os.makedirs(OBJ, exist_ok=True)
    headers = glob.glob(os.path.join(CSRC, "*.hpp")) + glob.glob(os.path.join(HERE, "..", "include", "*.h"))
    jobs = []
    objs = []
    for src, name, extra in units():
        obj = os.path.join(OBJ, name)
        objs.append(obj)
        if force or _stale(obj, [src] + headers):
            cmd = [cc, *FLAGS, *extra, "-c", src, "-o", obj]
            if keep_temps:
                cmd += ["-save-temps=obj"]
            jobs.append(cmd)

    if force or _stale(host_lib(), [HOST_SRC] + headers):
        jobs.append(host_command())

    def run(cmd):
        p = subprocess.run(cmd, capture_output=True, text=True)
        noise = "is not a recognized feature for this target"
        err = "\n".join(l for l in p.stderr.splitlines() if noise not in l)
        return p.returncode, cmd, err

    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, max(1, len(jobs)))) as ex:
        for rc, cmd, err in ex.map(run, jobs):
            if verbose and err.strip():
                print(err, file=sys.stderr)
            if rc != 0:
                raise RuntimeError("compilation failed: " + " ".join(cmd) + "\n" + err)
    if force or _stale(LIB, objs):
        cmd = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
        p = subprocess.run(cmd, capture_output=True, text=True)
        if p.returncode != 0:
            raise RuntimeError("link failed: " + p.stderr)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("--keep-temps", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force, keep_temps=a.keep_temps))
