"""Build libh3fp8.so (the HIP kernels + C ABI) for gfx950 with hipcc, and _host (the native host path of the common calls, a
CPython extension on the installed torch) with g++, in-tree.

    python minimax-h3-2x-dgx-spark-tp2_amd/build.py [--jobs N] [--asm]

Each csrc/*.hip compiles to an object under _build/ (git-ignored); the shared library lands next to the Python
package (h3_tp2_amd/libh3fp8.so), where the loader looks for it.  ``--asm`` also writes the gfx950 assembly of each
source to _build/ (for reading register use and the instruction schedule).
"""
from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "h3_tp2_amd", "libh3fp8.so")
HOST = os.path.join(HERE, "h3_tp2_amd", "_host" + sysconfig.get_config_var("EXT_SUFFIX"))
INCLUDE = os.path.join(os.path.dirname(HERE), "include")

ARCH = "gfx950"
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

# -packed-fp32-ops off: no v_pk_{add,mul,fma}_f32 anywhere; denormals kept; no contraction of a*b+c behind the
# reference's back (the epilogue's one fma is explicit).
COMMON = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-fno-gpu-flush-denormals-to-zero", "-ffp-contract=off",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    f"-I{INCLUDE}",
]


def sources() -> list[str]:
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str, asm: bool) -> str:
    obj = os.path.join(BUILD, os.path.basename(src)[:-4] + ".o")
    cmd = [HIPCC, *COMMON, "-c", src, "-o", obj]
    subprocess.run(cmd, check=True)
    if asm:
        s = os.path.join(BUILD, os.path.basename(src)[:-4] + f"-{ARCH}.s")
        subprocess.run([HIPCC, *COMMON, "--cuda-device-only", "-S", src, "-o", s], check=True)
    return obj


def build_host() -> str:
    """_host: csrc/host.cpp against torch's headers, linked to libh3fp8.so next to it."""
    import torch
    from torch.utils import cpp_extension
    root = os.environ.get("ROCM_PATH", "/opt/rocm")
    includes = [INCLUDE, *cpp_extension.include_paths(), sysconfig.get_paths()["include"], os.path.join(root, "include")]
    lib_dir = os.path.join(os.path.dirname(torch.__file__), "lib")
    tmp = HOST + ".tmp"
    subprocess.run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
                    f'-DH3_TORCH_VERSION="{torch.__version__}"',
                    f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", *(f"-I{d}" for d in includes),
                    os.path.join(CSRC, "host.cpp"), "-o", tmp, f"-L{os.path.dirname(LIB)}", "-lh3fp8", f"-L{lib_dir}",
                    "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python", "-Wl,-rpath,$ORIGIN"], check=True)
    os.replace(tmp, HOST)
    return HOST


def build(jobs: int = 4, asm: bool = False, verbose: bool = True) -> str:
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        objs = list(ex.map(lambda s: _compile(s, asm), srcs))
    tmp = LIB + ".tmp"
    subprocess.run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs], check=True)
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB} from {len(srcs)} sources", file=sys.stderr)
    try:
        build_host()
        if verbose:
            print(f"built {HOST}", file=sys.stderr)
    except (subprocess.CalledProcessError, OSError, ImportError) as e:      # no g++, no torch headers: Python does its work
        if os.path.exists(HOST):
            os.remove(HOST)                               # of an earlier library
        print(f"the library is built, {HOST} is not ({e}): its calls take the Python path", file=sys.stderr)
    return LIB


def main() -> None:
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    ap.add_argument("--asm", action="store_true")
    a = ap.parse_args()
    build(a.jobs, a.asm)


if __name__ == "__main__":
    main()
