"""Builds ``libllmmm.so`` (HIP kernels + C ABI) for gfx950 with hipcc and ``_native.so`` (the Python entry points' host work) with g++, in-tree.

``python llmmm_amd/build.py [--library]`` (run as a script: importing the package needs the libraries this
builds; ``--library``: ``libllmmm.so`` alone, without torch and g++).  hipcc cross-compiles without a GPU; the resulting libraries sit next to this file so
that they travel with the source tree.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OBJ = os.path.join(CSRC, "build")
LIB = os.path.join(HERE, "libllmmm.so")
BINDING = os.path.join(HERE, "_native.so")

COMMON = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
    # packed fp32 VALU ops are kept off for every device file
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]
# per-file extras: the FP8 kernels promote MFMA results with VALU FMAs, so the MFMA must
# write architectural VGPRs rather than AGPRs
SOURCES = {
    "fp16_gemm.hip": [],
    "fp8_gemm.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "fp8_skinny.hip": ["-mllvm", "-amdgpu-mfma-vgpr-form"],
    "quant_fp8.hip": [],
    "layout.hip": [],
    "probe.hip": [],
    "static_ws.hip": [],
    "capi.cpp": ["-x", "hip"],
}


def _compile(item):
    name, extra = item
    src = os.path.join(CSRC, name)
    obj = os.path.join(OBJ, os.path.splitext(name)[0] + ".o")
    cmd = ["hipcc"] + COMMON + extra + ["-c", src, "-o", obj]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "is not a recognized feature" not in l)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for %s:\n%s" % (name, out))
    return obj, out


def _compile_binding():
    """csrc/binding.cpp: host code only, against the headers of the installed torch and Python (g++)."""
    import sysconfig
    import torch
    obj = os.path.join(OBJ, "binding.o")
    cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-D_GLIBCXX_USE_CXX11_ABI=%d" % torch._C._GLIBCXX_USE_CXX11_ABI,
           "-I", sysconfig.get_paths()["include"], "-isystem", os.path.join(os.path.dirname(torch.__file__), "include"),
           "-c", os.path.join(CSRC, "binding.cpp"), "-o", obj]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("g++ failed for binding.cpp:\n" + res.stdout)
    return obj


def build(verbose=False):
    """Both libraries.  ``libllmmm.so`` needs hipcc only and is linked whether or not the Python side (g++, torch's headers) can be built."""
    os.makedirs(OBJ, exist_ok=True)
    with ThreadPoolExecutor(max_workers=5) as pool:
        binding = pool.submit(_compile_binding)
        build_library(pool, verbose)
        _link_binding(binding.result())
    return LIB


def build_library(pool, verbose=False):
    """``libllmmm.so``: all that a user of the C ABI or the C++ shims needs."""
    results = list(pool.map(_compile, SOURCES.items()))
    objs = [o for o, _ in results]
    if verbose:
        for _, out in results:
            if out.strip():
                print(out)
    cmd = ["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB] + objs
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout)


def _link_binding(obj):
    import torch
    torch_lib = os.path.join(os.path.dirname(torch.__file__), "lib")
    cmd = ["g++", "-shared", "-o", BINDING, obj, "-L", HERE, "-lllmmm", "-L", torch_lib, "-ltorch_python", "-ltorch_cpu", "-lc10", "-Wl,-rpath,$ORIGIN"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout)


def build_dropin_test():
    """Compile tests/cpp/dropin_test.cpp (the C++ drop-in shims of include/llmmm/mm) against the library."""
    root = os.path.dirname(HERE)
    src = os.path.join(root, "tests", "cpp", "dropin_test.cpp")
    out = os.path.join(root, "tests", "cpp", "dropin_test")
    cmd = ["hipcc", "-std=c++17", "-O1", "-Wno-unused-command-line-argument", "-I", os.path.join(root, "include"), "-o", out, src,
           "-L", HERE, "-lllmmm", "-Wl,-rpath,$ORIGIN/../../llmmm_amd"]
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        raise RuntimeError("hipcc failed for dropin_test.cpp:\n" + res.stdout)
    return out


if __name__ == "__main__":
    if "--library" in sys.argv:
        os.makedirs(OBJ, exist_ok=True)
        with ThreadPoolExecutor(max_workers=4) as library_pool:
            build_library(library_pool, verbose="-v" in sys.argv)
        print(LIB)
    else:
        print(build(verbose="-v" in sys.argv))
    print(build_dropin_test())
