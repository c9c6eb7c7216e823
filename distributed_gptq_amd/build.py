"""Builds libgptq_hip.so (the C-ABI library) in-tree for gfx950.

    python -m distributed_gptq_amd.build        # or __graft_entry__.build()

Every ``.hip``/``.cpp`` under ``csrc/`` is compiled with hipcc to an object
under ``csrc/_build/`` (in parallel) and linked into
``distributed_gptq_amd/libgptq_hip.so``; ``csrc/torch_ops.cc``, the native
torch operator over it, is compiled with g++ against torch's headers into
``distributed_gptq_amd/libgptq_torch.so``.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libgptq_hip.so")
TORCH_OUT = os.path.join(HERE, "libgptq_torch.so")
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON_FLAGS = [
    "-O3", "-fPIC", "-std=c++17", f"--offload-arch={ARCH}",
    "-mcode-object-version=5",
    # packed-fp32 instructions stay off (they have produced silent wrong
    # results on these boxes)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
    "-I", os.path.join(os.path.dirname(HERE), "include"),
]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC)
                  if f.endswith((".hip", ".cpp")))


def _compile(src, objdir, extra):
    obj = os.path.join(objdir, os.path.basename(src) + ".o")
    cmd = [HIPCC, *COMMON_FLAGS, *extra, "-c", src, "-o", obj]
    if src.endswith(".cpp"):
        cmd = [HIPCC, *COMMON_FLAGS, *extra, "-x", "hip", "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
    return obj, r.stderr


def build_torch_ops():
    """libgptq_torch.so (host code only; needs libgptq_hip.so to link)."""
    import torch
    base = os.path.dirname(torch.__file__)
    tmp = TORCH_OUT + ".tmp"
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-I", os.path.join(os.path.dirname(HERE), "include"), "-isystem", os.path.join(base, "include"),
           "-isystem", "/opt/rocm/include", os.path.join(CSRC, "torch_ops.cc"), "-o", tmp, "-L", HERE,
           "-l:libgptq_hip.so", "-L", os.path.join(base, "lib"), "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch",
           "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on torch_ops.cc:\n{r.stderr}")
    os.replace(tmp, TORCH_OUT)
    return TORCH_OUT


def build(verbose=False, extra=()):
    objdir = os.path.join(CSRC, "_build")
    os.makedirs(objdir, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        res = list(ex.map(lambda s: _compile(s, objdir, list(extra)), srcs))
    if verbose:
        for _, err in res:
            if err.strip():
                print(err, file=sys.stderr)
    tmp = OUT + ".tmp"
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp,
           *[o for o, _ in res]]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, OUT)
    build_torch_ops()
    return OUT


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
