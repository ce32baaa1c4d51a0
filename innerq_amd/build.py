"""Build libinnerq_hip.so in-tree with hipcc for gfx950, and the native call front _iqfast.so
(a CPython extension over libtorch, host code only) with the host compiler.

    python -m innerq_amd.build            # compile (always recompiles)

Every .hip source under innerq_amd/csrc is compiled to an object in parallel,
then linked into innerq_amd/libinnerq_hip.so.  Flags:

* ``--offload-arch=gfx950``: MI355X only, no other targets.
* ``-Xclang -target-feature -Xclang -packed-fp32-ops``: no packed-fp32 VALU
  forms (v_pk_{add,mul,fma}_f32) in any generated code.
* no fast-math: the quantizer relies on IEEE fp32 division and rounding.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libinnerq_hip.so")
FAST = os.path.join(HERE, "_iqfast.so")
OBJ_DIR = os.path.join(HERE, "_build")
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++20",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # matrix-core results in VGPRs: the GEMV epilogues read every MFMA result
    # with VALU instructions, which AGPR results would need copied out first
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wall",
    "-Wno-unused-function",
    "-Wno-unused-variable",
    "-Wno-unknown-pragmas",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; the HIP library cannot be built")


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src) + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr[-8000:]}")
    return obj


def build_fast() -> str:
    """csrc/iq_pyfast.cpp -> innerq_amd/_iqfast.so."""
    import sysconfig

    import torch
    t = os.path.dirname(torch.__file__)
    abi = int(torch._C._GLIBCXX_USE_CXX11_ABI)
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={abi}",
           f"-I{t}/include", f"-I{t}/include/torch/csrc/api/include", f"-I{sysconfig.get_paths()['include']}",
           os.path.join(CSRC, "iq_pyfast.cpp"), "-o", FAST + ".tmp", f"-L{t}/lib", "-ltorch_python", "-ltorch_cpu",
           "-lc10", f"-Wl,-rpath,{t}/lib"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"host compiler failed for iq_pyfast.cpp:\n{r.stderr[-8000:]}")
    os.replace(FAST + ".tmp", FAST)
    return FAST


def build(verbose: bool = True) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    jobs = max(1, min(len(srcs), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4))))
    with cf.ThreadPoolExecutor(jobs) as ex:
        fast = ex.submit(build_fast)
        objs = list(ex.map(_compile, srcs))
        fast.result()
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr[-8000:]}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    build()
