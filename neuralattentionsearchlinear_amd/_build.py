"""Builds csrc/*.hip into csrc/libnatsl.so for gfx950 with hipcc (cross-compiles without a GPU), and the benchmark's
clock probe (csrc/bench/) into csrc/libnatsl_bench.so, which is not part of the C ABI; and the layers' native host side
(csrc/host/, a Python module that sees torch's tensors) into _step_core.so."""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB = os.path.join(CSRC, "libnatsl.so")
BENCH_LIB = os.path.join(CSRC, "libnatsl_bench.so")
STEP_CORE = os.path.join(os.path.dirname(CSRC), "_step_core.so")
SOURCES = ["natsl_route.hip", "natsl_softmax.hip", "natsl_softmax_bwd.hip", "natsl_linear.hip", "natsl_linear_bwd.hip", "natsl_norm_gate.hip", "natsl_conv.hip", "natsl_decode.hip", "natsl_step.hip", "natsl_mixed.hip", "natsl_wgrad.hip", "natsl_project.hip", "natsl_narrow.hip", "natsl_front.hip", "natsl_cache.hip"]
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17",
    # keep the compiler from forming packed-fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    *os.environ.get("NATSL_HIPCC_EXTRA", "").split(),  # extra compiler flags for a development build
]


def _hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def _build_step_core():
    import torch
    from torch.utils.cpp_extension import include_paths
    srcs = [os.path.join(CSRC, "host", f) for f in ("step_core.cpp", "layer_core.cpp", "mixed_core.cpp")]
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-fPIC", "-shared", "-std=c++17", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           *(f"-I{d}" for d in (sysconfig.get_paths()["include"], *include_paths())), *srcs, "-o", STEP_CORE,
           "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-lc10", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compiling {srcs} failed:\n{r.stderr}")


def build(verbose: bool = False) -> str:
    hipcc = _hipcc()
    srcs = [s for s in SOURCES if os.path.exists(os.path.join(CSRC, s))]
    objs = []

    def compile_one(src):
        obj = os.path.join(CSRC, src.replace(".hip", ".o"))
        cmd = [hipcc, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
        if verbose and r.stderr.strip():
            print(r.stderr, file=sys.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=min(4, len(srcs))) as ex:
        step_core = ex.submit(_build_step_core)
        objs = list(ex.map(compile_one, srcs))
        step_core.result()
    r = subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    r = subprocess.run([hipcc, *FLAGS, "-shared", os.path.join(CSRC, "bench", "bench_probe.hip"), "-o", BENCH_LIB], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on bench/bench_probe.hip:\n{r.stderr}")
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
