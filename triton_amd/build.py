"""Build recipe for libtrinity_hip.so (hipcc, gfx950 only) and _host.so (g++), in-tree output.

    python -m triton_amd.build          # compile every csrc/*.hip and link; compile csrc/host/host.cpp against torch

Packed-FP32 VALU instructions are disabled for all device code (the flag below); the
host pass prints a harmless "unknown target feature" warning for it.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(HERE, "build")
LIB_PATH = os.path.join(HERE, "libtrinity_hip.so")
HOST_PATH = os.path.join(HERE, "_host.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-function",
    "-Wno-unknown-warning-option", "-Wno-unused-command-line-argument",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]
# What the compiler says of a kernel's registers, of which the build reports spills: several kernels here are shaped so that
# their registers just fit, and nothing but the time would tell otherwise.
RESOURCES = "-Rpass-analysis=kernel-resource-usage"
_SOURCE_LINE = re.compile(r"\s*\d* \| ")


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ_DIR, os.path.basename(src)[:-4] + ".o")
    cmd = [HIPCC, *FLAGS, RESOURCES, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    noise = "packed-fp32-ops' is not a recognized feature"
    kernel, skip = "", 0
    for line in r.stderr.splitlines():
        if f"[{RESOURCES}]" in line:                    # (two lines of source follow the first remark on a kernel)
            key, _, value = line.split("remark:", 1)[1].split(" [-R")[0].partition(": ")
            if key.strip() == "Function Name":
                kernel = value
            elif key.strip().startswith("ScratchSize") and int(value) > 0:
                sys.stderr.write(f"{os.path.basename(src)}: {kernel} spills: {value} bytes of scratch per lane\n")
            skip = 2
        elif skip and _SOURCE_LINE.match(line):
            skip -= 1
        elif line.strip() and noise not in line:
            sys.stderr.write(line + "\n")
    return obj


def build_host() -> str:
    """The host side of the modules (csrc/host/host.cpp): a CPython extension over torch's C++ tensors, linked to
    libtrinity_hip.so beside it."""
    import torch
    from torch.utils.cpp_extension import include_paths
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           *[f"-isystem{p}" for p in (*include_paths(), os.path.join(rocm, "include"), sysconfig.get_paths()["include"])],
           os.path.join(CSRC, "host", "host.cpp"), "-o", HOST_PATH, f"-L{lib}", "-lc10", "-lc10_hip", "-ltorch_cpu",
           "-ltorch_python", f"-L{HERE}", "-ltrinity_hip", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for host.cpp:\n{r.stdout}\n{r.stderr}")
    if r.stderr.strip():
        sys.stderr.write(r.stderr)
    return HOST_PATH


def build(verbose: bool = True, jobs: int = 6) -> str:
    os.makedirs(OBJ_DIR, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(jobs, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-Wl,--no-undefined", *objs, "-o", LIB_PATH]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    build_host()
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources, and {HOST_PATH}")
    return LIB_PATH


if __name__ == "__main__":
    build()
