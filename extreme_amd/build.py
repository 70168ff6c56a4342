"""Builds libxtreme_hip.so in-tree with hipcc for gfx950.

Each translation unit is compiled to an object in parallel, then linked into
extreme_amd/libxtreme_hip.so next to this file. Every HIP unit is compiled with packed FP32
instructions disabled (-target-feature -packed-fp32-ops).
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_obj")
LIB = os.path.join(HERE, "libxtreme_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"

SOURCES = ["op_fft_forward.hip", "op_fft_inverse.hip", "op_kernels.hip", "tensor_fft.hip",
           "krylov_kernels.hip", "green_assembly.hip", "obs_kernels.hip", "learned_kernels.hip", "probe_kernels.hip", "xtr_api.cpp"]
SOURCES += ["contract_direct.hip"]
SOURCES += [f"contract_block_{t}_{r}.hip" for t in ("c128", "c64") for r in "abcd"]

COMMON = ["-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
          "-I", os.path.join(HERE, "..", "include"), "-I", CSRC]


def _stale(src, out):
    """True when the object is missing or older than its source or any header in csrc/ and include/."""
    if not os.path.exists(out):
        return True
    deps = [os.path.join(CSRC, src)] + [os.path.join(CSRC, h) for h in os.listdir(CSRC) if h.endswith(".h")]
    inc = os.path.join(HERE, "..", "include")
    deps += [os.path.join(inc, h) for h in os.listdir(inc) if h.endswith(".h")]
    t = os.path.getmtime(out)
    return any(os.path.getmtime(d) > t for d in deps)


def _compile(src, incremental=False):
    out = os.path.join(OBJ, os.path.splitext(src)[0] + ".o")
    if incremental and not _stale(src, out):
        return out
    cmd = [HIPCC] + COMMON + ["-x", "hip", "-c", os.path.join(CSRC, src), "-o", out]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stderr}")
    return out


def build(verbose=False, incremental=False):
    """Compiles every unit (incremental=True recompiles only units older than their sources or the
    headers) and links the library."""
    os.makedirs(OBJ, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(lambda s: _compile(s, incremental), SOURCES))
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", LIB] + objs + ["-lpthread"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    if verbose:
        print(LIB)
    return LIB


if __name__ == "__main__":
    build(verbose=True, incremental="--incremental" in sys.argv)
    sys.exit(0)
