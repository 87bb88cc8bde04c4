"""Builds libsmlm_hip.so for gfx950 with hipcc (cross-compiles without a GPU) and the native host path with g++.

Usage: python -m loquetier_amd.build
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC_DIR = os.path.join(PKG_DIR, "csrc")
LIB_DIR = os.path.join(PKG_DIR, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libsmlm_hip.so")
HOST_PATH = os.path.join(LIB_DIR, "_smlm_host.so")  # Python extension: csrc/host_path.cpp
PROBE_PATH = os.path.join(LIB_DIR, "libsmlm_probe.so")
# library -> its translation units (headers are found through -I csrc)
LIBRARIES = {
    LIB_PATH: ["smlm_api.hip"],        # the operator library (include/smlm.h)
    PROBE_PATH: ["stream_probe.hip"],  # plain streaming kernels bench.py calibrates against
}

HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden",
    # keep the compiler from forming packed-fp32 VALU ops out of scalar float code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def hipcc_path() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.isabs(cand) and os.path.exists(cand) or not os.path.isabs(cand)):
            return cand
    return "hipcc"


def _compile(out: str, sources, verbose: bool) -> None:
    _run([hipcc_path(), *HIPCC_FLAGS, "-I", os.path.join(REPO_DIR, "include"), "-I", CSRC_DIR,
          *[os.path.join(CSRC_DIR, s) for s in sources], "-o", out + ".tmp"], out, verbose)


def _compile_host(out: str, verbose: bool) -> None:
    """The host path against the torch of this interpreter (host code only)."""
    import torch
    from torch.utils.cpp_extension import include_paths, library_paths
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", os.path.join(REPO_DIR, "include")]
    for inc in [*include_paths("cuda"), sysconfig.get_paths()["include"]]:
        cmd += ["-isystem", inc]
    cmd += [os.path.join(CSRC_DIR, "host_path.cpp"), "-o", out + ".tmp"]
    cmd += [f"-L{lib}" for lib in library_paths("cuda")]
    _run(cmd + ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip"], out, verbose)


def _run(cmd, out: str, verbose: bool) -> None:
    if verbose:
        print(" ".join(cmd), flush=True)
    res = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass warns that it does not know the packed-fp32 feature: harmless
    err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError(f"{os.path.basename(cmd[0])} failed ({res.returncode}):\n{err}")
    if err.strip() and verbose:
        print(err, file=sys.stderr)
    os.replace(out + ".tmp", out)


def build_library(verbose: bool = False) -> str:
    """Compile every HIP source into loquetier_amd/lib/ (always recompiles); returns the path of
    the operator library."""
    os.makedirs(LIB_DIR, exist_ok=True)
    for out, sources in LIBRARIES.items():
        _compile(out, sources, verbose)
    _compile_host(HOST_PATH, verbose)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(verbose=True))
