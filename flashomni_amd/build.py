"""Build the C-ABI library ``csrc/libflashomni_hip.so`` for gfx950 with hipcc, and the Python
extension ``_native.so`` on top of it with g++.

Usage: ``python -m flashomni_amd.build``.  hipcc cross-compiles without a GPU.
"""
import concurrent.futures
import os
import subprocess
import sys

CSRC = os.path.join(os.path.dirname(os.path.abspath(__file__)), "csrc")
LIB_PATH = os.path.join(CSRC, "libflashomni_hip.so")
NATIVE_PATH = os.path.join(os.path.dirname(CSRC), "_native.so")  # bindings.cpp: the Python API's call path
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
SOURCES = ["fo_error.cpp", "planner.cpp", "packbits.hip", "decode.hip", "sparse_fa.hip", "gemm.hip",
           "quant_fp8.hip", "symbols.hip"]
# -packed-fp32-ops off: the compiler must not form packed fp32 VALU instructions on this target
FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-x", "hip",
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-command-line-argument"]


def _compile(src, verbose):
    obj = os.path.join(CSRC, os.path.splitext(src)[0] + ".o")
    cmd = ["hipcc"] + FLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed on %s:\n%s" % (src, res.stderr))
    if verbose and res.stderr.strip():
        lines = [l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l]
        if lines:
            sys.stderr.write("\n".join(lines) + "\n")
    return obj


def _compile_native():
    """bindings.cpp -> object file: host code against torch's headers, no HIP compiler involved."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    obj = os.path.join(CSRC, "bindings.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-Wno-deprecated-declarations"]
    for inc in cpp_extension.include_paths() + [sysconfig.get_paths()["include"], os.path.join(ROCM, "include")]:
        cmd += ["-isystem", inc]
    res = subprocess.run(cmd + ["-c", os.path.join(CSRC, "bindings.cpp"), "-o", obj], capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed on bindings.cpp:\n%s" % res.stderr)
    return obj


def _link_native(obj):
    import torch
    lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-shared", "-o", NATIVE_PATH, obj, "-L" + CSRC, "-lflashomni_hip", "-L" + lib, "-ltorch_python", "-ltorch",
           "-ltorch_cpu", "-lc10", "-lc10_hip", "-lamdhip64", "-Wl,-rpath,$ORIGIN/csrc"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link of _native.so failed:\n%s" % res.stderr)


def build(verbose=False):
    """Compile every source (in parallel) and link the shared library and the extension.  Returns the
    library's path."""
    with concurrent.futures.ThreadPoolExecutor(max_workers=min(8, len(SOURCES) + 1)) as ex:
        native = ex.submit(_compile_native)
        objs = list(ex.map(lambda s: _compile(s, verbose), SOURCES))
    cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB_PATH] + objs
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n%s" % res.stderr)
    _link_native(native.result())
    return LIB_PATH


if __name__ == "__main__":
    print(build(verbose=True))
