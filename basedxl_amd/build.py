"""Builds libcascmm.so (HIP, gfx950 only) and _native.so (host C++) in-tree.

    python -m basedxl_amd.build

Every .hip file under csrc/ is one translation unit; they are compiled in parallel and
linked into basedxl_amd/libcascmm.so, which the ctypes loader in _lib.py opens.  csrc/host/native.cpp
becomes the extension module basedxl_amd._native, which takes ordinary eager calls to that library.
"""
from __future__ import annotations

import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libcascmm.so")
NATIVE = os.path.join(HERE, "_native.so")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", "--offload-arch=gfx950", "-fPIC",
    # packed fp32 VALU ops are kept out of the generated code on purpose
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def sources():
    return sorted(f for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(src: str) -> str:
    obj = os.path.join(OBJ, src[:-4] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "packed-fp32-ops" not in l and "warning generated" not in l)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def _compile_native() -> str:
    """The host extension's object (in a folder of its own: what lies beside it is the library's)."""
    import sysconfig

    import torch
    inc = os.path.join(os.path.dirname(torch.__file__), "include")
    obj = os.path.join(OBJ, "host", "native.o")
    os.makedirs(os.path.dirname(obj), exist_ok=True)
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-Wall", "-Wextra", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-isystem", inc, "-isystem", os.path.join(inc, "torch", "csrc", "api", "include"),
           "-isystem", "/opt/rocm/include", "-isystem", sysconfig.get_paths()["include"], "-c", os.path.join(CSRC, "host", "native.cpp"), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("g++ failed on native.cpp:\n" + r.stderr[-4000:])
    if r.stderr.strip():
        sys.stderr.write(r.stderr)
    return obj


def _link_native(obj: str) -> None:
    import torch
    libs = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", NATIVE, obj, "-L", libs, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_python",
           "-L", HERE, "-l:libcascmm.so", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link of _native.so failed:\n" + r.stderr)


def build(verbose: bool = True, jobs: int = 8) -> str:
    os.makedirs(OBJ, exist_ok=True)
    srcs = sources()
    with ThreadPoolExecutor(max_workers=min(jobs, len(srcs) + 1)) as ex:
        native = ex.submit(_compile_native)
        objs = list(ex.map(_compile, srcs))
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    # a kernel whose launch stub the compiler left out only shows up as an undefined symbol at load time
    import ctypes
    try:
        ctypes.CDLL(LIB)
    except OSError as e:
        raise RuntimeError(f"{LIB} was linked but does not load: {e}") from None
    _link_native(native.result())   # (behind the library, which also works without it)
    if verbose:
        print(f"built {LIB} from {len(srcs)} translation units, and {NATIVE}")
    return LIB


def _listing(src: str) -> str:
    """Assembly listing of one translation unit's device code (kept beside the objects, redone when a
    source under csrc/ is newer)."""
    out = os.path.join(OBJ, src[:-4] + ".gfx950.s")
    newest = max(os.path.getmtime(os.path.join(CSRC, f)) for f in os.listdir(CSRC) if f.endswith((".hip", ".h")))
    if not os.path.exists(out) or os.path.getmtime(out) < newest:
        os.makedirs(OBJ, exist_ok=True)
        tmp = f"{out}.{os.getpid()}.tmp"      # (another process may be making the same listing: rename a finished file into place)
        cmd = [HIPCC, *FLAGS, "-S", "--cuda-device-only", os.path.join(CSRC, src), "-o", tmp]
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            if os.path.exists(tmp):
                os.remove(tmp)
            raise RuntimeError(f"hipcc -S failed on {src}:\n{r.stderr[-2000:]}")
        os.replace(tmp, out)
    return out


def kernel_isa(symbol: str, jobs: int = 8) -> str:
    """gfx950 assembly of one kernel of the library, from its label to the end of its
    `.amdhsa_kernel` block (register counts, LDS and scratch sizes), compiled from the sources under
    csrc/ with the flags of the build.  `symbol` is what `cascmm_variant_kernel` or `cascmm_launched_kernel` returns."""
    srcs = [f for f in sources() if f.startswith("cascmm_inst_")] + [f for f in sources() if not f.startswith("cascmm_inst_")]
    with ThreadPoolExecutor(max_workers=min(jobs, len(srcs))) as ex:
        listings = list(ex.map(_listing, srcs))
    label, end = symbol + ":", ".end_amdhsa_kernel"
    for path in listings:
        with open(path) as f:
            text = f.read()
        at = text.find("\n" + label)
        if at < 0:
            continue
        meta = text.find("\t.amdhsa_kernel " + symbol + "\n", at)
        stop = text.find(end, meta if meta >= 0 else at)
        if stop < 0:
            continue
        return f"; {os.path.basename(path)}\n" + text[at + 1:stop + len(end)] + "\n"
    raise KeyError(f"no kernel {symbol} in the listings of {', '.join(srcs)}")


if __name__ == "__main__":
    build()
