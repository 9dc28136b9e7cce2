"""Compile libfmxq.so (the HIP kernels and the C ABI) in-tree for gfx950.

``python -m fastmlx_amd.build`` or ``fastmlx_amd.build.build()``.  Objects go to
``fastmlx_amd/_build/``; the shared library lands next to this file so it
travels with the source tree, and so does ``_fast``, the torch wrappers' call path, where
torch is installed.
``--diag`` (``build_diag()``) also builds the
time-line diagnostic program ``diag/qmv1_timeline``.
"""
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
CSRC = os.path.join(HERE, "csrc")
OUT_DIR = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libfmxq.so")
ARCH = os.environ.get("FMXQ_ARCH", "gfx950")

# -packed-fp32-ops keeps the compiler from emitting packed fp32 VALU ops.
HIP_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-Wall",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(HERE, "..", "include"),
]


def _hipcc() -> str:
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; libfmxq.so cannot be built")


def _compile(src: str, obj: str, flags=None) -> None:
    cmd = [_hipcc(), *(flags or HIP_FLAGS), "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    # hipcc's host pass warns that it does not know the packed-fp32 feature; drop that.
    noise = "is not a recognized feature for this target"
    msgs = [ln for ln in r.stderr.splitlines() if noise not in ln and ln.strip()]
    if msgs:
        print("\n".join(msgs), file=sys.stderr)


DIAG = os.path.join(HERE, "diag")
TIMELINE = os.path.join(DIAG, "qmv1_timeline")


def build_diag(verbose: bool = True) -> str:
    """The time-line diagnostic (diag/qmv1_timeline.hip): a program, not part of the
    library, linked with its own build of fmxq_qmv.hip under FMXQ_QMV1_TIMELINE."""
    os.makedirs(OUT_DIR, exist_ok=True)
    flags = [*HIP_FLAGS, "-I", CSRC, "-DFMXQ_QMV1_TIMELINE"]
    objs = []
    for src in (os.path.join(DIAG, "qmv1_timeline.hip"), os.path.join(CSRC, "fmxq_qmv.hip")):
        obj = os.path.join(OUT_DIR, "timeline_" + os.path.basename(src) + ".o")
        _compile(src, obj, flags)
        objs.append(obj)
    r = subprocess.run([_hipcc(), f"--offload-arch={ARCH}", "-o", TIMELINE, *objs],
                       capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {TIMELINE}\n{r.stdout}\n{r.stderr}")
    if verbose:
        print(f"built {TIMELINE}")
    return TIMELINE


# Tagged with the interpreter's ABI, so another Python in the same tree does not load it.
FAST = os.path.join(HERE, "_fast" + sysconfig.get_config_var("EXT_SUFFIX"))


def _cxx() -> str | None:
    rocm = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "llvm", "bin", "clang++")
    return shutil.which("g++") or shutil.which("clang++") or (rocm if os.path.exists(rocm) else None)


def build_fast(verbose: bool = True) -> str | None:
    """The torch wrappers' call path in C++ (ext/fmxq_fast.cpp), a CPython module linked
    against torch and the libfmxq.so next to it.  The wrappers run without it, so where
    torch for ROCm or a C++ compiler is missing it is left out and None returned."""
    spec = importlib.util.find_spec("torch")
    torch_dir = list(spec.submodule_search_locations)[0] if spec else ""
    lib = os.path.join(torch_dir, "lib")
    cxx = _cxx()
    old = os.path.join(HERE, "_fast.so")  # the name without a tag, from an earlier build
    if os.path.exists(old):
        os.remove(old)
    if not cxx or not os.path.exists(os.path.join(lib, "libc10_hip.so")):
        if verbose:
            print("skipped " + FAST + ": " + ("no torch for ROCm" if cxx else "no C++ compiler"))
        return None
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    inc = [os.path.join(torch_dir, "include"), sysconfig.get_paths()["include"],
           os.path.join(torch_dir, "include", "torch", "csrc", "api", "include"),
           os.path.join(rocm, "include")]
    tmp = FAST + ".tmp"
    cmd = [cxx, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-D__HIP_PLATFORM_AMD__=1",
           "-DUSE_ROCM=1", *(a for d in inc for a in ("-isystem", d)),
           os.path.join(HERE, "ext", "fmxq_fast.cpp"), "-o", tmp, f"-L{lib}", "-lc10", "-lc10_hip",
           "-ltorch_cpu", "-ltorch_python", f"-L{HERE}", "-l:libfmxq.so", "-Wl,-rpath,$ORIGIN",
           f"-Wl,-rpath,{lib}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"compile failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, FAST)
    if verbose:
        print(f"built {FAST}")
    return FAST


def build(verbose: bool = True) -> str:
    os.makedirs(OUT_DIR, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")) + glob.glob(os.path.join(CSRC, "*.cpp")))
    objs = [os.path.join(OUT_DIR, os.path.basename(s) + ".o") for s in srcs]
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        list(ex.map(_compile, srcs, objs))
    tmp = LIB + ".tmp"
    rocm_lib = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "lib")
    cmd = [_hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs,
           f"-L{rocm_lib}", f"-Wl,-rpath,{rocm_lib}"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed: {' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    build_fast(verbose)
    return LIB


if __name__ == "__main__":
    build()
    if "--diag" in sys.argv[1:]:
        build_diag()
