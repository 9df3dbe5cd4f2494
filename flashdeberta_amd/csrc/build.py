"""Build libfdb_hip.so (gfx950) with hipcc and the host extension _native.so with the C++ compiler, in-tree.

    python -m flashdeberta_amd.csrc.build

The shared objects land next to the package (flashdeberta_amd/libfdb_hip.so, flashdeberta_amd/_native.so) so that
they travel with the source tree; nothing is installed outside it.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(HERE)
LIB = os.path.join(PKG, "libfdb_hip.so")
NATIVE = os.path.join(PKG, "_native.so")
SOURCES = ["fdb_api.cpp", "fdb_attn.hip", "fdb_near.hip", "fdb_near_f32.hip", "fdb_small.hip", "fdb_fp8.hip", "fdb_aux.hip", "fdb_bwd.hip", "fdb_bwd_ring.hip", "fdb_chain.hip", "fdb_linear.hip", "fdb_gemm.hip", "fdb_grad.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950", "-x", "hip",
    # packed fp32 VALU forms are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _compile(src):
    obj = os.path.join(HERE, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC, *FLAGS, "-c", os.path.join(HERE, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    err = "\n".join(l for l in r.stderr.splitlines() if "is not a recognized feature for this target" not in l)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (src, err))
    return obj, err


def _compile_native():
    """csrc/fdb_torch.cpp: host code only, against torch's headers; it finds libfdb_hip.so beside itself."""
    import torch

    base = os.path.dirname(torch.__file__)
    obj = os.path.join(HERE, "fdb_torch.o")
    rocm = os.path.dirname(os.path.dirname(HIPCC))
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-c", os.path.join(HERE, "fdb_torch.cpp"), "-o", obj,
           "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
           "-isystem", os.path.join(base, "include"), "-isystem", os.path.join(base, "include", "torch", "csrc", "api", "include"),
           "-isystem", os.path.join(rocm, "include"), "-isystem", sysconfig.get_paths()["include"]]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("the C++ compiler failed for fdb_torch.cpp:\n" + r.stderr)
    return obj, os.path.join(base, "lib")


def _link_native(obj, torch_lib):
    cmd = [os.environ.get("CXX", "g++"), "-shared", "-o", NATIVE, obj, "-L" + PKG, "-l:libfdb_hip.so", "-Wl,-rpath,$ORIGIN",
           "-L" + torch_lib, "-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-lhipblaslt"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    os.remove(obj)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)


def build(verbose=True):
    with ThreadPoolExecutor(max_workers=len(SOURCES) + 1) as ex:
        native = ex.submit(_compile_native)
        results = list(ex.map(_compile, SOURCES))
        native_obj, torch_lib = native.result()
    objs = [o for o, _ in results]
    for _, err in results:
        if verbose and err.strip():
            print(err, file=sys.stderr)
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIB, *objs]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stderr)
    for o in objs:
        os.remove(o)
    _link_native(native_obj, torch_lib)
    if verbose:
        print("built", LIB, NATIVE)
    return LIB


if __name__ == "__main__":
    build()
