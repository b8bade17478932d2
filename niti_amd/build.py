"""Builds niti_amd/libniti_gfx950.so from niti_amd/csrc/*.hip with hipcc for gfx950.

Usage: ``python -m niti_amd.build`` (cross-compiles without a GPU present)."""
from __future__ import annotations

import concurrent.futures as cf
import glob
import importlib.util
import os
import shutil
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "build")
SO = os.path.join(HERE, "libniti_gfx950.so")
HOST_SO = os.path.join(HERE, "_host.so")      # the tensor front end, a Python module

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
    # keep the compiler from forming packed-fp32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    cmd = [HIPCC, *FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed on %s:\n%s\n%s" % (src, r.stdout, r.stderr))
    return obj


def _host_flags() -> tuple:
    """Compiler and linker flags of the tensor front end: torch's headers and libraries, found without importing torch."""
    torch_dir = os.path.join(importlib.util.find_spec("torch").submodule_search_locations[0])
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    inc = [os.path.join(ROOT, "include"), os.path.join(torch_dir, "include"), os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"),
           os.path.join(rocm, "include"), sysconfig.get_paths()["include"]]
    lib = os.path.join(torch_dir, "lib")
    return (["-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM", "-Wno-deprecated-declarations"] + ["-I" + d for d in inc],
            ["-L" + HERE, "-l:libniti_gfx950.so", "-L" + lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python",
             "-L" + os.path.join(rocm, "lib"), "-lamdhip64", "-Wl,-rpath,$ORIGIN", "-Wl,-rpath," + lib])


def _compile_host(src: str) -> str:
    obj = os.path.join(OBJ, os.path.basename(src) + ".o")
    r = subprocess.run(["g++", *_host_flags()[0], "-c", src, "-o", obj], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed on %s:\n%s\n%s" % (src, r.stdout, r.stderr))
    return obj


def build(verbose: bool = False) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    if not srcs:
        raise RuntimeError("no HIP sources under " + CSRC)
    host_srcs = sorted(glob.glob(os.path.join(CSRC, "host", "*.cpp")))
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + len(host_srcs))) as ex:
        host = [ex.submit(_compile_host, s) for s in host_srcs]
        objs = list(ex.map(_compile, srcs))
        host_objs = [h.result() for h in host]
    tmp = SO + ".tmp"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (r.stdout, r.stderr))
    # a shared library links with undefined symbols left in it: resolve them all now, in a child process, so that
    # a library that cannot be loaded is never installed
    chk = subprocess.run([sys.executable, "-c", "import ctypes, os, sys; ctypes.CDLL(sys.argv[1], mode=os.RTLD_NOW)", tmp],
                         capture_output=True, text=True)
    if chk.returncode != 0:
        os.unlink(tmp)
        raise RuntimeError("the linked library does not load:\n" + chk.stderr[-2000:])
    os.replace(tmp, SO)
    tmp = HOST_SO + ".tmp"
    r = subprocess.run(["g++", "-shared", "-o", tmp, *host_objs, *_host_flags()[1]], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n%s\n%s" % (r.stdout, r.stderr))
    os.replace(tmp, HOST_SO)
    if verbose:
        print("built", HOST_SO, os.path.getsize(HOST_SO), "bytes")
        print("built", SO, os.path.getsize(SO), "bytes")
    return SO


if __name__ == "__main__":
    build(verbose=True)
    sys.exit(0)
