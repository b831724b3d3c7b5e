"""Builds libca_hip.so (hipcc for gfx950) and _ca_torch.so (the torch binding of
its autograd functions, host code only) in-tree.

Usage: python continuum-attention_amd/build.py [--verbose]
The shared libraries are written next to this file and loaded by _native.py.
"""
from __future__ import annotations

import concurrent.futures
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libca_hip.so")
SOURCES = ["ca_fwd.hip", "ca_bwd.hip", "ca_bwd_dkdv.hip", "ca_weights.hip", "ca_norm.hip",
           "ca_optim.hip", "ca_swiglu.hip", "ca_abi.hip", "ca_noalloc.hip"]
ARCH = os.environ.get("CA_OFFLOAD_ARCH", "gfx950")
TORCH_SOURCE = "ca_torch.cpp"
TORCH_EXT = os.path.join(HERE, "_ca_torch.so")

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=fast",
    # packed fp32 VALU forms are disabled: some of them have returned wrong
    # results on this GPU with no error
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # keep MFMA accumulators in VGPRs: the dK/dV kernel otherwise shuffles
    # loop-carried tiles between AGPRs every iteration (~100 moves per tile)
    "-mllvm", "-amdgpu-mfma-vgpr-form",
    "-Wall",
    "-Wno-unused-function",
]


# The attention kernels compute no output from a NaN or infinity they form
# themselves (the backward's fast-path segment math may form one in lane 0,
# which has no left neighbour, and discards it), so they are built assuming
# finite values, which lets fmax/fmin skip canonicalisation.  NaN or infinite
# inputs still propagate through their arithmetic (tests pin that).  The
# other sources (norms, optimizer, SwiGLU, weight rows) keep IEEE semantics:
# a diverging run's non-finite values must behave there as in torch.
_FINITE_MATH = ["-fno-honor-nans", "-fno-honor-infinities"]
# The attention kernels contract multiply-adds only within one source
# expression (their fused multiply-adds are written as fmaf): every template
# instantiation (fp32, bf16, fp16 operands; each head dim) then rounds the same
# arithmetic the same way, so the bf16 forward, which skips the zero limb
# products of bf16-valued operands, returns the fp32 forward's results on the
# same values bit for bit.  Measured: the same instruction counts in the tile
# loops as contraction across statements.
_ATTN = _FINITE_MATH + ["-ffp-contract=on"]

SOURCE_FLAGS = {"ca_fwd.hip": _ATTN, "ca_bwd.hip": _ATTN, "ca_bwd_dkdv.hip": _ATTN}


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC)")


def _jobs() -> int:
    # at most 8 compiles at once (one per source; hipcc is single-threaded)
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    return max(1, min(8, n, len(SOURCES)))


def _run(cmd, what: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"{what} failed:\n{res.stdout}{res.stderr}")


def compile_torch_ext(obj: str, verbose: bool) -> None:
    """ca_torch.cpp against the installed torch's headers (host code only)."""
    import sysconfig

    import torch
    from torch.utils.cpp_extension import include_paths
    inc = [*include_paths(), sysconfig.get_paths()["include"], "/opt/rocm/include"]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-DTORCH_EXTENSION_NAME=_ca_torch",
          "-DTORCH_API_INCLUDE_EXTENSION_H", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          *(x for d in inc for x in ("-isystem", d)), "-c", os.path.join(CSRC, TORCH_SOURCE),
          "-o", obj], f"g++ on {TORCH_SOURCE}", verbose)


def link_torch_ext(obj: str, verbose: bool) -> None:
    from torch.utils.cpp_extension import library_paths
    tmp = TORCH_EXT + ".tmp"
    _run(["g++", "-shared", obj, "-o", tmp, *(f"-L{d}" for d in library_paths()), "-ltorch",
          "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_python", f"-L{HERE}",
          "-l:" + os.path.basename(LIB), "-Wl,-rpath,$ORIGIN"], "torch binding link", verbose)
    os.replace(tmp, TORCH_EXT)


def build(verbose: bool = False, extra_flags=None) -> str:
    build_dir = os.path.join(HERE, "_build")
    os.makedirs(build_dir, exist_ok=True)
    flags = HIPCC_FLAGS + list(extra_flags or [])

    def compile_one(src):
        obj = os.path.join(build_dir, src.replace(".hip", ".o"))
        cmd = [hipcc(), *flags, *SOURCE_FLAGS.get(src, []), "-c", os.path.join(CSRC, src), "-o", obj]
        res = subprocess.run(cmd, capture_output=True, text=True)
        out = "\n".join(l for l in (res.stdout + res.stderr).splitlines()
                        if "packed-fp32-ops" not in l)
        return src, cmd, obj, res.returncode, out

    objs = []
    ext_obj = os.path.join(build_dir, TORCH_SOURCE.replace(".cpp", ".o"))
    with concurrent.futures.ThreadPoolExecutor(_jobs()) as pool:
        ext = pool.submit(compile_torch_ext, ext_obj, verbose)
        for src, cmd, obj, rc, out in pool.map(compile_one, SOURCES):
            if verbose:
                print(" ".join(cmd), flush=True)
            if rc != 0:
                raise RuntimeError(f"hipcc failed on {src}:\n{out}")
            if verbose and out.strip():
                print(out, flush=True)
            objs.append(obj)
    tmp = LIB + ".tmp"
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}{res.stderr}")
    os.replace(tmp, LIB)
    ext.result()  # the C library stands also where g++ or torch's headers are missing
    link_torch_ext(ext_obj, verbose)
    return LIB


if __name__ == "__main__":
    print(build(verbose="--verbose" in sys.argv))
