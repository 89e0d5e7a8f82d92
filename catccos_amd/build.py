"""Builds libcatccos_mx.so (HIP kernels + C ABI) for gfx950 with hipcc, and the extension of the Python front end with g++.

Usage: python -m catccos_amd.build [--verbose] [--jobs N]
Objects go to catccos_amd/_build/, the library to catccos_amd/lib/.  Sources are
rebuilt when they or any header are newer than the object (``force`` rebuilds all).
"""
from __future__ import annotations

import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "libcatccos_mx.so")
NATIVE_SRC = os.path.join(CSRC, "native_call.cpp")
# the name carries the interpreter's ABI tag, so that another Python looks for an extension of its own
NATIVE = os.path.join(HERE, "_native_call" + sysconfig.get_config_var("EXT_SUFFIX"))

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"), "-I" + CSRC,
    "-Wno-unused-command-line-argument",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _headers_mtime() -> float:
    hs = [os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".h")]
    hs.append(os.path.join(ROOT, "include", "catccos_mx.h"))
    return max(os.path.getmtime(h) for h in hs)


def _filter(text: str) -> str:
    keep = [ln for ln in text.splitlines()
            if "packed-fp32-ops' is not a recognized feature" not in ln and ln.strip()]
    return "\n".join(keep)


def compile_object(path: str, obj: str, extra_flags=(), verbose: bool = False) -> str:
    """hipcc -c of one .hip file with the library's flags (plus ``extra_flags``)."""
    cmd = [HIPCC, *FLAGS, *extra_flags, "-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = _filter(r.stdout + r.stderr)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {path}:\n{out}")
    if verbose and out:
        print(out)
    return obj


def link_shared(lib: str, objs) -> str:
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", lib, *objs],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + _filter(r.stdout + r.stderr))
    return lib


def _compile(src: str, verbose: bool) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    out = _filter(r.stdout + r.stderr)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{out}")
    if verbose and out:
        print(out)
    return obj


def build_native(force: bool = False) -> str:
    """The Python extension catccos_amd._native_call (host code only, against this interpreter's torch).  It reads torch's structures, so
    it is rebuilt when torch, Python or the command changes (the stamp beside the objects), not only for a newer source."""
    import torch
    t = os.path.dirname(torch.__file__)
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           f'-DCMX_TORCH_VERSION="{torch.__version__}"', "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM",
           "-isystem", os.path.join(t, "include"), "-isystem", os.path.join(t, "include", "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(ROCM, "include"), "-isystem", sysconfig.get_paths()["include"], NATIVE_SRC,
           "-L" + os.path.join(t, "lib"), "-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip", "-ltorch_hip"]
    stamp, want = os.path.join(OBJ, "native_call.stamp"), "\n".join([sys.version, *cmd])
    if (not force and os.path.exists(NATIVE) and os.path.getmtime(NATIVE) >= os.path.getmtime(NATIVE_SRC)
            and os.path.exists(stamp) and open(stamp).read() == want):
        return NATIVE
    # to a file of its own, moved into place when it is whole: a build that is interrupted or runs twice leaves no part of one
    tmp = f"{NATIVE}.{os.getpid()}"
    r = subprocess.run([*cmd, "-o", tmp], capture_output=True, text=True)
    if r.returncode != 0:
        if os.path.exists(tmp):
            os.remove(tmp)
        raise RuntimeError(f"g++ failed on {NATIVE_SRC}:\n" + r.stdout + r.stderr)
    os.replace(tmp, NATIVE)
    os.makedirs(OBJ, exist_ok=True)
    with open(stamp, "w") as f:
        f.write(want)
    return NATIVE


def build(force: bool = False, verbose: bool = False, jobs: int = 4) -> str:
    os.makedirs(OBJ, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    build_native(force)
    hm = _headers_mtime()
    todo, objs = [], []
    for s in sources():
        obj = os.path.join(OBJ, s[:-4] + ".o")
        objs.append(obj)
        stale = (force or not os.path.exists(obj)
                 or os.path.getmtime(obj) < max(os.path.getmtime(os.path.join(CSRC, s)), hm))
        if stale:
            todo.append(s)
    with ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        list(ex.map(lambda s: _compile(s, verbose), todo))
    if todo or not os.path.exists(LIB):
        r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs],
                           capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("link failed:\n" + _filter(r.stdout + r.stderr))
    return LIB


if __name__ == "__main__":
    force = "--force" in sys.argv
    verbose = "--verbose" in sys.argv
    print(build(force=force, verbose=verbose))
