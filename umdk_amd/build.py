"""Builds libcamhip.so (the C-ABI library of HIP kernels for gfx950) in-tree.

    python -m umdk_amd.build              # -> umdk_amd/lib/libcamhip.so, umdk_amd/_camcall.so

Every source is compiled by hipcc for gfx950 only; symbols are hidden except
the extern "C" entry points declared in include/camhip.h.  _camcall.so is the
Python caller of those entry points (host code, g++); it takes them from the library that _lib has loaded.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libcamhip.so")
CALLER = os.path.join(HERE, "_camcall.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # packed fp32 vector ops stay disabled: some of their forms gave wrong results on this GPU pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"), "-Wall", "-Wno-unused-result",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith((".hip", ".cpp")))


def _compile(src, defines=(), build_dir=BUILD):
    obj = os.path.join(build_dir, src + ".o")
    cmd = [HIPCC] + COMMON + list(defines) + ["-c", os.path.join(CSRC, src), "-o", obj]
    if src.endswith(".cpp"):
        cmd[1:1] = ["-x", "hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = "\n".join(l for l in (r.stdout + r.stderr).splitlines() if "packed-fp32-ops" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{msgs}")
    if msgs.strip():
        print(msgs, file=sys.stderr)
    return obj


def _build_caller():
    tmp = CALLER + ".tmp"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-fvisibility=hidden", "-Wall",
           "-I" + os.path.join(ROOT, "include"), "-I" + sysconfig.get_paths()["include"],
           os.path.join(HERE, "pyext", "camcall.cpp"), "-o", tmp, "-ldl"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building _camcall.so failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, CALLER)


def build(verbose=True, defines=(), lib=LIB):
    """Compile every source and link `lib`.  `defines` (e.g. ["-DCAM_GMM_TIMELINE"]) build a variant,
    with its objects in a build folder of its own."""
    build_dir = BUILD if not defines else os.path.join(BUILD, "variant_" + "_".join(d.lstrip("-D") for d in defines))
    os.makedirs(build_dir, exist_ok=True)
    os.makedirs(os.path.dirname(lib), exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(lambda f: _compile(f, defines, build_dir), srcs))
    tmp = lib + ".tmp"
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, lib)
    if lib == LIB:
        _build_caller()
    if verbose:
        print(f"built {lib}")
    return lib


if __name__ == "__main__":
    build()
