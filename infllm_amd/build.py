"""Build libinfllm_hip.so (gfx950) with hipcc and the extension module _host.so with the host compiler, in-tree.

    python -m infllm_amd.build

The library is cross-compiled (no GPU needed).  Both are placed next to this file so
that they travel with the source tree.
"""
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB_PATH = os.path.join(HERE, "libinfllm_hip.so")
HOST_PATH = os.path.join(HERE, "_host.so")
SOURCES = ["abi.hip", "ingest.hip", "attn.hip", "score.hip", "retrieve.hip", "decode.hip", "window.hip", "cache.hip", "stream.hip", "resident.hip"]
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc_path():
    for cand in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    proc = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass reports that it does not know the packed-fp32 feature; that is expected
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in proc.stderr.splitlines() if noise not in l)
    if proc.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed:\n" + err)
    if verbose and err.strip():
        print(err, file=sys.stderr)


def _library(out, verbose, extra_flags):
    # ROCr (libhsa-runtime64) is linked for the DMA-engine copy of carved units; in a process it is the copy the HIP
    # runtime already loaded
    _run([hipcc_path(), *HIPCC_FLAGS, *extra_flags, *[os.path.join(CSRC, s) for s in SOURCES], "-o", out, "-lhsa-runtime64"], verbose)


def _host_module(out, verbose):
    """csrc/host.cpp against the installed torch.  (Its libraries are in the process when the module is imported: no path to them.)"""
    import torch
    from torch.utils import cpp_extension
    cxx = os.environ.get("CXX") or shutil.which("g++") or shutil.which("c++")
    if not cxx:
        raise RuntimeError("no C++ compiler found (set CXX)")
    include = [sysconfig.get_paths()["include"], *cpp_extension.include_paths()]
    _run([cxx, "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
          f'-DINFLLM_TORCH_VERSION="{torch.__version__}"', *[f"-I{p}" for p in include],
          os.path.join(CSRC, "host.cpp"), "-o", out, *[f"-L{p}" for p in cpp_extension.library_paths()], "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10"],
         verbose)


def build(verbose=True, extra_flags=()):
    """Both, or neither: they share include/infllm_hip.h, and one that failed leaves the pair that was there."""
    new = {path: path[:-len(".so")] + ".new.so" for path in (LIB_PATH, HOST_PATH)}
    try:
        _library(new[LIB_PATH], verbose, extra_flags)
        _host_module(new[HOST_PATH], verbose)
        for path, made in new.items():
            os.replace(made, path)
    finally:
        for made in new.values():
            if os.path.exists(made):
                os.remove(made)
    return LIB_PATH


if __name__ == "__main__":
    print(build())
