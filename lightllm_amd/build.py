"""Compiles the HIP sources under csrc/ into lib/libmi355fp8.so for gfx950 with hipcc, and its CPython entry beside it."""
import importlib.machinery
import os
import shutil
import subprocess
import sys
import sysconfig

_HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(_HERE, "csrc")
LIB_DIR = os.path.join(_HERE, "lib")
LIB_PATH = os.path.join(LIB_DIR, "libmi355fp8.so")
CALL_PATH = os.path.join(LIB_DIR, "_mi355call" + importlib.machinery.EXTENSION_SUFFIXES[0])
SOURCES = ["capi.hip", "group_quant.hip", "weight_quant.hip", "block_gemm.hip", "rows128_few.hip", "rows128_some.hip", "rows128_many.hip", "linear.hip", "moe_align.hip", "moe_elementwise.hip", "routed_ffn.hip", "probe.hip"]
# packed-fp32 VALU ops are switched off for every kernel of this library
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def build(verbose: bool = False) -> str:
    """Always recompiles (object per source, then link); returns the library path."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(LIB_DIR, "obj")
    os.makedirs(obj_dir, exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES:
        path = os.path.join(CSRC, src)
        if not os.path.exists(path):
            continue
        obj = os.path.join(obj_dir, src.replace(".hip", ".o"))
        objs.append(obj)
        cmd = [hipcc] + FLAGS + ["-c", path, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)))
    failed = False
    for src, p in procs:
        out, _ = p.communicate()
        out = "\n".join(l for l in out.splitlines() if "is not a recognized feature for this target" not in l)
        if p.returncode != 0:
            failed = True
            print(f"[build] {src} FAILED\n{out}", file=sys.stderr)
        elif verbose and out.strip():
            print(out)
    if failed:
        raise RuntimeError("hipcc failed")
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH] + objs
    subprocess.check_call(cmd)
    _build_call(verbose)
    return LIB_PATH


def _build_call(verbose: bool) -> None:
    """The CPython entry.  It is linked against nothing (it gets the address of the C entry), and where the interpreter's headers or
    a C compiler are missing it is left out: the package calls through ctypes then."""
    if os.path.exists(CALL_PATH):
        os.remove(CALL_PATH)
    include = sysconfig.get_paths()["include"]
    cc = next((c for c in (os.environ.get("CC"), "gcc", "cc", "clang") if c and shutil.which(c.split()[0])), None)
    if cc is None or not os.path.exists(os.path.join(include, "Python.h")):
        print(f"[build] no {'C compiler' if cc is None else 'Python.h'}: the one-call linear goes through ctypes", file=sys.stderr)
        return
    cmd = cc.split() + ["-O2", "-Wall", "-Wextra", "-shared", "-fPIC", "-I" + include, os.path.join(CSRC, "pycall.c"), "-o", CALL_PATH]
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.check_call(cmd)


if __name__ == "__main__":
    print(build(verbose=True))
