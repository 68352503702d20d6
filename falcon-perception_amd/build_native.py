"""Build libfp_paged_kv.so (the gfx950 kernels + C ABI) with hipcc, and fp_host.so (its calls from PyTorch tensors) with g++, in-tree.

    python falcon-perception_amd/build_native.py

hipcc cross-compiles for gfx950 without a GPU.  The kernels' library has no torch
or Python dependency; the host package loads it with ctypes.  fp_host.so is a Python module on top of it.
"""

from __future__ import annotations

import concurrent.futures
import os
import re
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
OUT_DIR = os.path.join(HERE, "falcon_perception_amd", "_lib")
LIB_PATH = os.path.join(OUT_DIR, "libfp_paged_kv.so")
HOST_PATH = os.path.join(OUT_DIR, "fp_host.so")
OBJ_DIR = os.path.join(HERE, "build")

# packed-FP32 VALU forms are switched off for every kernel of this library
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    # one remark per kernel with its registers, LDS and scratch: kept beside the object file
    # (build/<source>.resources.txt) and read back by `resource_usage()`
    "-Rpass-analysis=kernel-resource-usage",
    "-I", INCLUDE,
    "-I", CSRC,
]


def _hipcc() -> str:
    exe = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
    if not os.path.exists(exe):
        raise RuntimeError("hipcc not found; the ROCm toolchain is required to build libfp_paged_kv.so")
    return exe


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    cmd = [_hipcc(), *FLAGS, "-c", src, "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{res.stdout}\n{res.stderr}")
    with open(obj[:-2] + ".resources.txt", "w") as f:
        f.write(res.stderr)
    return obj


def resource_usage() -> dict[str, dict[str, int]]:
    """Per kernel of the last build: {"vgprs", "agprs", "scratch" (bytes per lane), "lds" (bytes per workgroup),
    "occupancy" (wavefronts per SIMD), "sgprs_moved" (scalar registers kept in lanes of vector registers)}, keyed by the mangled kernel name; builds first if nothing has been
    built.  A kernel with scratch > 0 spills registers to memory; the first launch of such a kernel makes the
    runtime set that memory up, which it cannot do while a stream is being captured into a graph."""
    names = [os.path.join(OBJ_DIR, os.path.basename(s)[:-4] + ".resources.txt") for s in sources()]
    if not all(os.path.exists(n) for n in names):
        build_library(verbose=False)
    out: dict[str, dict[str, int]] = {}
    fields = {"vgprs": r"VGPRs: (\d+)", "agprs": r"AGPRs: (\d+)", "scratch": r"ScratchSize \[bytes/lane\]: (\d+)",
              "lds": r"LDS Size \[bytes/block\]: (\d+)", "occupancy": r"Occupancy \[waves/SIMD\]: (\d+)",
              "sgprs_moved": r"SGPRs Spill: (\d+)"}
    for n in names:
        with open(n) as f:
            text = f.read()
        for block in re.split(r"remark: [^\n]*Function Name: ", text)[1:]:
            out[block.split()[0]] = {k: int(re.search(v, block).group(1)) for k, v in fields.items()}
    return out


def _compile_host() -> str:
    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(OBJ_DIR, "host.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-I", INCLUDE,
           "-I", sysconfig.get_paths()["include"]]
    for path in cpp_extension.include_paths():
        cmd += ["-isystem", path]
    res = subprocess.run([*cmd, "-c", os.path.join(CSRC, "host.cpp"), "-o", obj], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{res.stdout}\n{res.stderr}")
    return obj


def _link_host(obj: str) -> None:
    import torch

    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST_PATH + ".tmp"
    res = subprocess.run(["g++", "-shared", obj, "-o", tmp, "-L", OUT_DIR, "-l:" + os.path.basename(LIB_PATH), "-Wl,-rpath,$ORIGIN",
                          "-L", libs, "-ltorch_python", "-ltorch_cpu", "-lc10"], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link of fp_host.so failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, HOST_PATH)


def build_library(verbose: bool = True) -> str:
    """Compile every csrc/*.hip for gfx950 and link libfp_paged_kv.so, and fp_host.so on top of it. Returns the library's path."""
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(OUT_DIR, exist_ok=True)
    srcs = sources()
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(_compile_host)
        objs = list(ex.map(_compile, srcs))
    tmp = LIB_PATH + ".tmp"
    cmd = [_hipcc(), "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", tmp]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    _link_host(host.result())
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build_library()
