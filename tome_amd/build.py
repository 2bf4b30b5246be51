"""Build recipe for libtome_logprob.so (hipcc, gfx950 only) and _torch_ops.so (its host side for torch tensors, g++)."""
from __future__ import annotations

import os
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_PATH = os.path.join(PKG_DIR, "libtome_logprob.so")
OPS_PATH = os.path.join(PKG_DIR, "_torch_ops.so")
SOURCES = [*(f"fused_dma_{k}{o}.hip" for o in ("entropy_argmax", "entropy", "argmax", "plain") for k in ("any_", "")),
           "fused_lmhead.hip", "capi.hip", "row_logprob.hip", "row_sample.hip", "full_log_softmax.hip", "lora_merge.hip", "mfma_probe.hip"]

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fno-gpu-rdc",
    # hipcc -O3 would otherwise form packed-fp32 instructions from ordinary float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _run(cmd: list[str], verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass warns that it does not know the packed-fp32 feature; drop that noise
    err = "\n".join(l for l in proc.stderr.splitlines() if "packed-fp32-ops" not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed ({proc.returncode}): {' '.join(cmd)}\n{err}")
    if verbose and err.strip():
        print(err, file=sys.stderr)


def build_torch_ops(verbose: bool = False) -> str:
    """The host side of the tensor operators: plain C++ against torch's headers (no GPU code), linked to the library
    beside it."""
    import sysconfig

    import torch
    from torch.utils import cpp_extension
    cxx = os.environ.get("CXX", "g++")
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    _run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
          f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          *[f"-I{d}" for d in cpp_extension.include_paths()], f"-I{sysconfig.get_paths()['include']}",
          os.path.join(CSRC, "torch_binding.cpp"), "-o", OPS_PATH, f"-L{torch_lib}", "-lc10", "-ltorch_cpu", "-ltorch_python",
          f"-L{PKG_DIR}", "-l:libtome_logprob.so", "-Wl,-rpath,$ORIGIN"], verbose)
    return OPS_PATH


def build(verbose: bool = False, extra_flags: list[str] | None = None, out: str | None = None) -> str:
    """Compile every HIP source (one hipcc process per file, side by side) and link the in-tree shared library;
    returns its path.  Objects go to a temporary directory and nothing but the library is left behind.  With the default ``out`` the
    tensor operators' host side is built after it."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    out = out or LIB_PATH
    flags = HIPCC_FLAGS + list(extra_flags or [])
    jobs = max(1, min(len(SOURCES), int(os.environ.get("MAX_JOBS", os.cpu_count() or 1))))
    with tempfile.TemporaryDirectory(prefix="tome_build_") as tmp:
        objs = [os.path.join(tmp, s.replace(".hip", ".o")) for s in SOURCES]
        with ThreadPoolExecutor(max_workers=jobs) as pool:
            list(pool.map(lambda so: _run([hipcc, *flags, "-c", os.path.join(CSRC, so[0]), "-o", so[1]], verbose),
                          zip(SOURCES, objs)))
        _run([hipcc, "--offload-arch=gfx950", "-fPIC", "-shared", "-fno-gpu-rdc", "-o", out, *objs], verbose)
    if out == LIB_PATH:
        build_torch_ops(verbose)
    return out


if __name__ == "__main__":
    print(build(verbose=True, extra_flags=sys.argv[1:]))
