"""Builds ``libbam_hip.so`` (the HIP kernels + C ABI) for gfx950 with hipcc, and ``_bam_host.so`` (the native host layer
on top of it, a torch extension module) with the host compiler.

The library has no dependency on torch or Python: plain ``hipcc -shared``.  Both are built
in-tree, next to this file, so that the very same binaries are what tests, the smoke check
and the benchmark load.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG_DIR, "csrc")
LIB_PATH = os.path.join(PKG_DIR, "libbam_hip.so")
HOST_PATH = os.path.join(PKG_DIR, "_bam_host.so")
# the longest compilations first: they are spread over the workers
SOURCES = ["bwd_long.hip", "bwd_dkdv.hip", "bwd_dkdv_save.hip", "bwd_dq_saved.hip", "bwd_dq.hip", "bwd_both.hip", "fwd_long.hip", "fwd.hip", "tile_flags.hip", "decode.hip", "bam_abi.hip"]
ARCH = "gfx950"
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-fno-gpu-rdc",
    # no NaN is ever produced on purpose (masked scores are -inf, never NaN), so max/min need no
    # NaN-quieting canonicalisation instructions
    "-fno-honor-nans",
    # packed fp32 VALU ops are kept off for all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found: libbam_hip.so cannot be built")


def _rocm_include() -> str:
    return os.path.join(os.path.dirname(os.path.dirname(os.path.realpath(_hipcc()))), "include")


def _compile_host(objdir: str) -> str:
    """host.cpp -> object file (it includes torch's headers, which takes longer than most kernel files)."""
    import sysconfig

    from torch.utils import cpp_extension

    obj = os.path.join(objdir, "host.o")
    includes = [f"-I{p}" for p in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"])]
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wno-attributes", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-I{_rocm_include()}", "-DTORCH_API_INCLUDE_EXTENSION_H",
           "-DTORCH_EXTENSION_NAME=_bam_host", *includes, "-c", os.path.join(CSRC, "host.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed on host.cpp:\n{r.stderr}")
    return obj


def _link_host(obj: str) -> None:
    from torch.utils import cpp_extension

    libs = [f"-L{p}" for p in cpp_extension.library_paths()]
    tmp = HOST_PATH + ".tmp"
    cmd = ["g++", "-shared", "-o", tmp, obj, f"-L{PKG_DIR}", "-lbam_hip", "-Wl,-rpath,$ORIGIN", *libs, "-lc10", "-lc10_hip",
           "-ltorch", "-ltorch_cpu", "-ltorch_python"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link of the host layer failed:\n{r.stderr}")
    os.replace(tmp, HOST_PATH)


def build_library(force: bool = True, verbose: bool = False) -> str:
    """Compile every kernel file and the host layer and link both.  Returns the path of the HIP library."""
    if not force and os.path.exists(LIB_PATH) and os.path.exists(HOST_PATH):
        return LIB_PATH
    hipcc = _hipcc()
    objdir = os.path.join(PKG_DIR, "build")
    os.makedirs(objdir, exist_ok=True)

    def compile_one(src: str) -> str:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmd = [hipcc, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{r.stderr}")
        if verbose:
            sys.stderr.write(r.stderr)
        return obj

    with ThreadPoolExecutor(max_workers=min(len(SOURCES) + 1, os.cpu_count() or 4)) as ex:
        host = ex.submit(_compile_host, objdir)
        objs = list(ex.map(compile_one, SOURCES))
        host_obj = host.result()
    tmp = LIB_PATH + ".tmp"
    r = subprocess.run([hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host_obj)
    return LIB_PATH


if __name__ == "__main__":
    print(build_library(force=True, verbose="-v" in sys.argv))
