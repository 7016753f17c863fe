"""Builds libd2conv.so (the C-ABI HIP library) for gfx950 with hipcc, and _native.so (its torch binding) with g++.

    python -m d2conv3d_amd.build [--force]

Each csrc/*.hip is compiled to an object under csrc/build/ and the objects are
linked into d2conv3d_amd/libd2conv.so; no torch headers are involved there.
"""
import concurrent.futures
import glob
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libd2conv.so")

HIPCC = os.environ.get("HIPCC") or shutil.which("hipcc") or "/opt/rocm/bin/hipcc"
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-fPIC", "-std=c++17", "-munsafe-fp-atomics",
    # packed-FP32 instructions are kept out of the generated code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function",
]


def _newer(src, dst, deps):
    if not os.path.exists(dst):
        return True
    t = os.path.getmtime(dst)
    return any(os.path.getmtime(p) > t for p in [src] + deps)


def _compile(src, force):
    obj = os.path.join(OBJ, os.path.basename(src)[:-4] + ".o")
    deps = glob.glob(os.path.join(CSRC, "*.hpp")) + [os.path.join(HERE, "..", "include", "d2conv.h")]
    if force or _newer(src, obj, deps):
        cmd = [HIPCC] + FLAGS + ["-c", src, "-o", obj]
        r = subprocess.run(cmd, capture_output=True, text=True)
        noise = "is not a recognized feature for this target"
        err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
        if r.returncode != 0:
            raise RuntimeError(f"hipcc failed for {src}:\n{err}")
        if err.strip():
            sys.stderr.write(err + "\n")
    return obj


def build_library(force=False, jobs=8):
    os.makedirs(OBJ, exist_ok=True)
    srcs = sorted(glob.glob(os.path.join(CSRC, "*.hip")))
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        objs = list(ex.map(lambda s: _compile(s, force), srcs))
    if force or not os.path.exists(LIB) or any(os.path.getmtime(o) > os.path.getmtime(LIB) for o in objs):
        cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError(f"link failed:\n{r.stderr}")
    return LIB


NATIVE_SRC = os.path.join(CSRC, "torch", "native.cpp")
NATIVE = os.path.join(HERE, "_native.so")


def build_native(force=False):
    """The torch binding (host code only), linked to the library beside it."""
    if not (force or _newer(NATIVE_SRC, NATIVE, [os.path.join(HERE, "..", "include", "d2conv.h")])):
        return NATIVE
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    rocm = os.path.dirname(os.path.dirname(os.path.realpath(HIPCC)))
    if not os.path.exists(os.path.join(rocm, "include", "hip")):
        rocm = "/opt/rocm"
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
           f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}",
           f"-I{root}/include", f"-I{root}/include/torch/csrc/api/include", f"-I{rocm}/include", f"-I{sysconfig.get_paths()['include']}",
           NATIVE_SRC, "-o", NATIVE, f"-L{root}/lib", "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip", f"-L{HERE}",
           "-ld2conv", f"-L{rocm}/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"{cmd[0]} failed for {NATIVE_SRC}:\n{r.stderr}")
    return NATIVE


if __name__ == "__main__":
    print(build_library(force="--force" in sys.argv))
    print(build_native(force="--force" in sys.argv))
