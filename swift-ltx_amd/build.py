"""Build the gfx950 shared libraries in-tree with hipcc.

    python swift-ltx_amd/build.py            # rebuild every object
    python swift-ltx_amd/build.py --if-stale # only when a source is newer

csrc/*.hip -> lib/libswiftltx_q4.so, the drop-in library (include/swiftltx_q4.h).
csrc/bench/*.hip -> lib/libswiftltx_bench.so, measurement kernels that only
bench.py loads (the HBM read ceiling); not part of the C ABI.
csrc/py/q4_binding.cpp -> lib/_q4_binding.<Python ABI>.torch-<version>.so, the
native marshalling of the Python mirror's hot calls (a CPython extension over
torch's C++ tensors; host code, built with g++ where torch is installed).  It
reads tensors through torch's inlined accessors, so it serves only the Python
and the torch that it was built against: its name holds both, and the mirror
looks for the name of its own.  The mirror works without it (through ctypes),
so where it cannot be built the libraries still are, with a warning.
Objects go to swift-ltx_amd/_build/, the libraries to swift-ltx_amd/lib/.
Every HIP file is compiled for gfx950 only, with packed-fp32 instruction
selection disabled (hipcc's host pass warns that it does not know the
feature; that warning is expected).
"""
from __future__ import annotations

import concurrent.futures as cf
import glob
import importlib.util
import os
import re
import shutil
import subprocess
import sys
import sysconfig

PKG = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
OBJ_DIR = os.path.join(PKG, "_build")
LIB_DIR = os.path.join(PKG, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libswiftltx_q4.so")
BENCH_LIB_PATH = os.path.join(LIB_DIR, "libswiftltx_bench.so")
BINDING_SRC = os.path.join(CSRC, "py", "q4_binding.cpp")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

DEVICE_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I" + os.path.join(REPO, "include"),
]


def sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def bench_sources() -> list[str]:
    return sorted(glob.glob(os.path.join(CSRC, "bench", "*.hip")))


def headers() -> list[str]:
    return (sorted(glob.glob(os.path.join(CSRC, "*.hpp")))
            + sorted(glob.glob(os.path.join(REPO, "include", "*.h"))))


def _older(outputs: list[str], inputs: list[str]) -> bool:
    if not all(os.path.exists(f) for f in outputs):
        return True
    t = min(os.path.getmtime(f) for f in outputs)
    return any(os.path.getmtime(f) > t for f in inputs)


def libs_stale() -> bool:
    return _older([LIB_PATH, BENCH_LIB_PATH], sources() + bench_sources() + headers() + [__file__])


def binding_stale() -> bool:
    path = binding_path()
    return path is not None and _older([path], headers() + [BINDING_SRC, __file__])


def torch_dir() -> str | None:
    """The installed torch's folder, found without importing it."""
    spec = importlib.util.find_spec("torch")
    return os.path.dirname(spec.origin) if spec and spec.origin else None


def binding_path() -> str | None:
    """The binding's path for this Python and the installed torch (None without
    one): the name __init__.py looks for.  Of torch, the version and the commit,
    read from its version.py."""
    t = torch_dir()
    if not t or not os.path.exists(os.path.join(t, "version.py")):
        return None
    text = open(os.path.join(t, "version.py")).read()
    version, commit = (re.search(rf"^{k}\b[^=\n]*=\s*'([^']*)'", text, re.M)
                       for k in ("__version__", "git_version"))
    if not version:
        return None
    return os.path.join(LIB_DIR, "_q4_binding.%s.torch-%s-%s.so" % (
        sysconfig.get_config_var("SOABI"), version[1], commit[1][:8] if commit else ""))


def _build_binding(path: str) -> None:
    t = torch_dir()
    tmp = path + ".tmp%d" % os.getpid()
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           "-I" + os.path.join(REPO, "include"), "-I" + os.path.join(t, "include"),
           "-I" + os.path.join(t, "include", "torch", "csrc", "api", "include"),
           "-I" + sysconfig.get_paths()["include"],
           "-isystem", os.path.join(os.path.dirname(os.path.dirname(shutil.which(HIPCC) or HIPCC)), "include"),
           BINDING_SRC, "-o", tmp, "-L" + os.path.join(t, "lib"),
           "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"g++ failed for {BINDING_SRC}:\n{r.stderr}")
    os.replace(tmp, path)


def _compile(src: str) -> str:
    sub = "bench_" if os.path.basename(os.path.dirname(src)) == "bench" else ""
    obj = os.path.join(OBJ_DIR, sub + os.path.basename(src) + ".o")
    cmd = [HIPCC, *DEVICE_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _link(objs: list[str], path: str) -> None:
    tmp = path + ".tmp%d" % os.getpid()
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", tmp, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    os.replace(tmp, path)


def build(force: bool = True, jobs: int = 8) -> str:
    """Compile every csrc/*.hip (and csrc/bench/*.hip) for gfx950, link
    LIB_PATH and BENCH_LIB_PATH, and build the binding where that can be done;
    returns LIB_PATH."""
    path = binding_path()
    libs, binding = force or libs_stale(), path is not None and (force or binding_stale())
    if not libs and not binding:
        return LIB_PATH
    os.makedirs(OBJ_DIR, exist_ok=True)
    os.makedirs(LIB_DIR, exist_ok=True)
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        built = ex.submit(_build_binding, path) if binding else None
        if libs:
            main, bench = sources(), bench_sources()
            objs = list(ex.map(_compile, main + bench))
            _link(objs[:len(main)], LIB_PATH)
            _link(objs[len(main):], BENCH_LIB_PATH)
    try:
        if built is not None:
            built.result()
    except (RuntimeError, OSError) as e:
        # no g++, Python headers or ROCm torch, say
        built = None
        sys.stderr.write(f"warning: {path} not built, ctypes serves every call: {e}\n")
    # Bindings of other builds, and one that could not be built again, may not
    # fit the library.
    for old in glob.glob(os.path.join(LIB_DIR, "_q4_binding*.so")):
        if old != path or (binding and built is None):
            os.remove(old)
    return LIB_PATH


if __name__ == "__main__":
    stale_only = "--if-stale" in sys.argv
    print(build(force=not stale_only))
