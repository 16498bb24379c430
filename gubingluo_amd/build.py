"""Build recipe of librtm_hip.so (gfx950) and the rtm_gpu drop-in driver.

    python -m gubingluo_amd.build        # or __graft_entry__.build()

Everything is compiled in-tree with hipcc; outputs:
    gubingluo_amd/librtm_hip.so   the C-ABI library (include/rtm_hip.h)
    gubingluo_amd/rtm_gpu         the drop-in driver executable (RTM_GPU_velstr.cpp's role)
"""
from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "librtm_hip.so")
EXE = os.path.join(PKG, "rtm_gpu")
ARCH = os.environ.get("RTM_OFFLOAD_ARCH", "gfx950")

HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-result", "-Wno-unused-function",
]
LIB_SOURCES = ["rtm_kernels.hip", "rtm_engine.cpp", "rtm_server.cpp", "rtm_capi.cpp", "host_io.cpp",
               "host_driver.cpp", "field_data.cpp", "postprocess_noalloc.hip"]


def _hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found")


def _run(cmd):
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = (r.stdout + r.stderr)
    # the host pass does not know the gfx target feature; harmless
    out = "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{out}")
    return out


def build_library(verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    hipcc = _hipcc()
    objs = []
    jobs = []
    for src in LIB_SOURCES:
        s = os.path.join(CSRC, src)
        o = os.path.join(BUILD, src.rsplit(".", 1)[0] + ".o")
        objs.append(o)
        lang = ["-x", "hip"]
        jobs.append([hipcc, *lang, *HIP_FLAGS, "-I", os.path.join(ROOT, "include"), "-c", s, "-o", o])
    with ThreadPoolExecutor(max_workers=min(8, len(jobs))) as ex:
        for out in ex.map(_run, jobs):
            if verbose and out.strip():
                print(out)
    tmp = LIB + ".tmp"
    _run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs, "-lpthread"])
    os.replace(tmp, LIB)
    return LIB


def build_driver() -> str:
    hipcc = _hipcc()
    src = os.path.join(CSRC, "rtm_gpu_main.cpp")
    tmp = EXE + ".tmp"
    _run([hipcc, "-O2", "-std=c++17", "-I", os.path.join(ROOT, "include"), "-I", CSRC, src, "-o", tmp,
          "-L", PKG, "-lrtm_hip", f"-Wl,-rpath,$ORIGIN"])
    os.replace(tmp, EXE)
    return EXE


def build_oracle() -> None:
    d = os.path.join(ROOT, "oracle")
    _run(["make", "-C", d, "-s", "-B", "liboracle.so"])
    if os.path.exists("/root/reference/FD_function.cpp"):   # an empty folder: fixtures stay as committed
        _run(["make", "-C", d, "-s", "-B", "ref"])


def build_all(verbose: bool = False) -> None:
    build_library(verbose)
    build_driver()
    build_oracle()


if __name__ == "__main__":
    build_all(verbose="-v" in sys.argv)
    print("built", LIB, EXE)
