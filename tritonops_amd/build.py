"""Build libmi_attn.so (HIP kernels + C ABI) for gfx950 with plain hipcc, and
_native.so (the host side of the usual calls, linked to it and to torch) with g++.

Usage: python -m tritonops_amd.build [--jobs N] [--keep-temps]
Both are written next to this file so that they travel with the package.
"""
import argparse
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ_DIR = os.path.join(CSRC, "build")
LIB_PATH = os.path.join(HERE, "libmi_attn.so")
SOURCES = ["api.cpp", "bench_timing.cpp", "prefill.hip", "decode.hip", "bwd.hip", "rmsnorm.hip", "xent.hip", "xent_grad.hip", "transpose.hip"]
NATIVE_SRC = os.path.join(CSRC, "host_calls.cpp")
NATIVE_PATH = os.path.join(HERE, "_native.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
CXX = os.environ.get("CXX", "g++")
FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    # packed-FP32 VALU forms are kept out of every kernel of this library
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _compile(src, extra):
    obj = os.path.join(OBJ_DIR, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, "-x", "hip", *FLAGS, *extra, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, err))
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _native_object():
    """host_calls.cpp: host code only, against torch's and Python's headers."""
    import torch
    from torch.utils import cpp_extension

    obj = os.path.join(OBJ_DIR, "host_calls.o")
    include = cpp_extension.include_paths() + [sysconfig.get_paths()["include"]]
    cmd = [CXX, "-O2", "-std=c++17", "-fPIC", "-Wall", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
           '-DMI_TORCH_VERSION="%s"' % torch.__version__, '-DMI_PYTHON_VERSION="%d.%d"' % sys.version_info[:2],
           *("-isystem" + i for i in include), "-c", NATIVE_SRC, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("%s failed for host_calls.cpp:\n%s" % (CXX, r.stderr))
    if r.stderr.strip():
        sys.stderr.write(r.stderr)
    return obj, cpp_extension.library_paths()


def _link_native(obj, lib_dirs):
    cmd = [CXX, "-shared", "-o", NATIVE_PATH, obj, "-L" + HERE, "-l:" + os.path.basename(LIB_PATH), "-Wl,-rpath,$ORIGIN",
           *("-L" + d for d in lib_dirs), "-ltorch_python", "-ltorch_cpu", "-lc10"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)


def build(jobs=4, keep_temps=False, verbose=True):
    os.makedirs(OBJ_DIR, exist_ok=True)
    extra = ["-save-temps=obj"] if keep_temps else []
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(_native_object)
        objs = list(ex.map(lambda s: _compile(s, extra), SOURCES))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    _link_native(*native.result())
    if verbose:
        print("built", LIB_PATH, NATIVE_PATH)
    return LIB_PATH


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=4)
    ap.add_argument("--keep-temps", action="store_true")
    a = ap.parse_args()
    build(a.jobs, a.keep_temps)
