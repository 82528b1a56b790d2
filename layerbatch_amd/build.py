"""Build liblbmoe.so (gfx950) and the host extension in-tree.

    python -m layerbatch_amd.build   # compile every csrc/*.hip, link liblbmoe.so; build _host.so

Objects go to layerbatch_amd/_build/, the library to layerbatch_amd/liblbmoe.so (hipcc, with
packed-fp32 instruction generation disabled), the CPython extension of csrc/host_ext.cpp, which
uses torch's C++ tensors, to layerbatch_amd/_host.so (the host compiler).
"""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys
import sysconfig
import warnings

PKG = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(PKG, "csrc")
BUILD = os.path.join(PKG, "_build")
LIB = os.path.join(PKG, "liblbmoe.so")
HOST = os.path.join(PKG, "_host.so")
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}", "-O3", "-fPIC", "-std=c++20", "-Wall",
    "-Wno-unused-function", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (set HIPCC or install ROCm)")


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _compile(hipcc, src):
    obj = os.path.join(BUILD, os.path.basename(src)[:-4] + ".o")
    cmd = [hipcc, *HIPCC_FLAGS, "-c", src, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{r.stdout}\n{r.stderr}")
    noise = "is not a recognized feature for this target"
    warn = "\n".join(l for l in r.stderr.splitlines() if noise not in l and l.strip())
    return obj, warn


def _host_cxx(hipcc):
    """A host C++ compiler: CXX, the system's, or the clang++ that hipcc itself runs; or None."""
    near = os.path.dirname(os.path.realpath(hipcc))
    for cand in (os.environ.get("CXX"), "g++", "c++", os.path.join(near, "amdclang++"),
                 os.path.join(near, "..", "llvm", "bin", "clang++"), "clang++"):
        path = shutil.which(cand) if cand else None
        if path:
            return path
    return None


def _build_host(hipcc):
    """Compile and link the host extension against the installed torch. Without a host compiler or
    Python's headers none is left in place: the module calls then take the general Python path."""
    import torch
    cxx = _host_cxx(hipcc)
    python_h = os.path.join(sysconfig.get_paths()["include"], "Python.h")
    if not cxx or not os.path.exists(python_h):
        warnings.warn("the host extension is not built: "
                      + ("no host C++ compiler found (set CXX)" if not cxx else f"no {python_h}"),
                      RuntimeWarning, stacklevel=2)
        if os.path.exists(HOST):
            os.remove(HOST)
        return
    root = os.path.dirname(torch.__file__)
    inc, rocm = os.path.join(root, "include"), os.environ.get("ROCM_PATH", "/opt/rocm")
    tmp = HOST + ".tmp"
    cmd = [cxx, "-O2", "-fPIC", "-std=c++17", "-shared", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
           "-I" + inc, "-I" + os.path.join(inc, "torch", "csrc", "api", "include"),
           "-I" + os.path.join(rocm, "include"), "-I" + sysconfig.get_paths()["include"],
           os.path.join(CSRC, "host_ext.cpp"), "-o", tmp, "-L" + os.path.join(root, "lib"),
           "-ltorch_python", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"host extension build failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, HOST)


def build(verbose=False):
    """Compile all sources, link liblbmoe.so and build the host extension. Returns the library
    path."""
    hipcc = _hipcc()
    os.makedirs(BUILD, exist_ok=True)
    srcs = sources()
    with cf.ThreadPoolExecutor(max_workers=min(8, len(srcs) + 1)) as ex:
        host = ex.submit(_build_host, hipcc)
        results = list(ex.map(lambda s: _compile(hipcc, s), srcs))
        host.result()
    for obj, warn in results:
        if warn and verbose:
            print(warn, file=sys.stderr)
    tmp = LIB + ".tmp"
    cmd = [hipcc, f"--offload-arch={ARCH}", "-shared", "-fPIC", *[o for o, _ in results], "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stdout}\n{r.stderr}")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose=True))
