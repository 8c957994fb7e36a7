"""Build recipe for libwan_attn.so, the gfx950 HIP kernels behind include/wan_attn.h, and for
libwan_ops-torch<version>.so, the torch operators' native kernels that call it (host code).

Each csrc/*.hip file is compiled with hipcc for gfx950 only, in parallel, and
the objects are linked into one shared library next to this file (in-tree, so
it travels with the source tree to the machine that runs it).  Packed fp32
VALU instructions are disabled for all device code.  csrc/torch_ops.cpp is
compiled with the host compiler against the installed torch.

Usage: python wan2-ti2v-5b_amd/build.py [--clean]
"""
import concurrent.futures as cf
import os
import shutil
import subprocess
import sys

PKG_DIR = os.path.dirname(os.path.abspath(__file__))
REPO_DIR = os.path.dirname(PKG_DIR)
CSRC = os.path.join(PKG_DIR, "csrc")
BUILD_DIR = os.path.join(PKG_DIR, "_build")
LIB_NAME = "libwan_attn.so"
LIB_PATH = os.path.join(PKG_DIR, LIB_NAME)
ARCH = "gfx950"

HIPCC = os.environ.get("HIPCC", os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc"))
DEVICE_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    # no packed fp32 VALU ops (v_pk_fma_f32 / v_pk_mul_f32 / v_pk_add_f32)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(REPO_DIR, "include"),
]


def sources():
    return sorted(os.path.join(CSRC, f) for f in os.listdir(CSRC) if f.endswith(".hip"))


def _run(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    # hipcc's host pass warns that it does not know the packed-fp32 feature; that is expected.
    out = "\n".join(l for l in p.stdout.splitlines()
                    if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"build failed ({' '.join(cmd)}):\n{out}")
    return out


def _ops_lib_path():
    """The torch operators' library: named for the torch that it is built against, which alone loads it."""
    import torch
    return os.path.join(PKG_DIR, f"libwan_ops-torch{torch.__version__}.so")


def _ops_commands(obj, out):
    """Compile and link commands of the torch operators."""
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include")]
    cxx = os.environ.get("CXX", "g++")
    compile_ = [cxx, "-O2", "-std=c++17", "-fPIC", "-Wall", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
                f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
                *[a for i in inc for a in ("-isystem", i)], "-c", os.path.join(CSRC, "torch_ops.cpp"), "-o", obj]
    link = [cxx, "-shared", obj, "-o", out, "-L", PKG_DIR, f"-l:{LIB_NAME}", "-L", os.path.join(root, "lib"),
            "-lc10", "-ltorch_cpu", "-lc10_hip", "-ltorch_hip", "-Wl,-rpath,$ORIGIN"]
    return compile_, link


def build(verbose: bool = False) -> str:
    """Compile every HIP source and link libwan_attn.so, then the operators' library; returns the path of the first."""
    if not os.path.exists(HIPCC):
        raise RuntimeError(f"hipcc not found at {HIPCC}")
    os.makedirs(BUILD_DIR, exist_ok=True)
    srcs = sources()
    objs = [os.path.join(BUILD_DIR, os.path.basename(s) + ".o") for s in srcs]
    jobs = min(len(srcs) + 1, int(os.environ.get("MAX_JOBS", "8")))
    with cf.ThreadPoolExecutor(max_workers=max(1, jobs)) as ex:
        futs = [ex.submit(_run, [HIPCC, *DEVICE_FLAGS, "-c", s, "-o", o]) for s, o in zip(srcs, objs)]
        ops_path = _ops_lib_path()
        ops_tmp = ops_path + ".tmp"
        compile_ops, link_ops = _ops_commands(os.path.join(BUILD_DIR, "torch_ops.o"), ops_tmp)
        futs.append(ex.submit(_run, compile_ops))
        for f in futs:
            out = f.result()
            if verbose and out.strip():
                print(out)
    tmp = LIB_PATH + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp])
    os.replace(tmp, LIB_PATH)
    _run(link_ops)
    for f in os.listdir(PKG_DIR):
        if f.startswith("libwan_ops") and f.endswith(".so"):      # of older sources, or for another torch
            os.remove(os.path.join(PKG_DIR, f))
    os.replace(ops_tmp, ops_path)
    if verbose:
        print(f"built {LIB_PATH} and {os.path.basename(ops_path)}")
    return LIB_PATH


if __name__ == "__main__":
    if "--clean" in sys.argv:
        shutil.rmtree(BUILD_DIR, ignore_errors=True)
    build(verbose=True)
