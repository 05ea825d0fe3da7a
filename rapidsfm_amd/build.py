"""Builds librsfm_amd.so (HIP, gfx950) in-tree with hipcc.

Usage: python rapidsfm_amd/build.py  (or __graft_entry__.build()).
Every source is compiled with contraction of multiply-add off, so the FP32
RANSAC kernels round exactly like their CPU restatement, and with the
packed-FP32 instructions disabled.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
LIB = os.path.join(HERE, "librsfm_amd.so")
OBJDIR = os.path.join(HERE, "_build")

SOURCES = [
    "api.cpp",
    "bf_match.hip",
    "bf_aux.hip",
    "ransac.hip",
    "ransac_finish.hip",
    "cashash.hip",
    "rmf.hip",
    "mlp.hip",
    "pipeline.hip",
    "degensac.hip",
    "pose.hip",
    "undistort.hip",
]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("RSFM_OFFLOAD_ARCH", "gfx950")

COMMON = [
    "-O3", "-fPIC", "-std=c++17", "-Wall", "-Wno-unused-function",
    "-ffp-contract=off", "-fno-fast-math",
    "-I" + INCLUDE, "-I" + CSRC,
]
DEVICE = [
    "--offload-arch=" + ARCH,
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-munsafe-fp-atomics",
]


def _defines():
    # optional tile-configuration overrides, e.g. RSFM_DEFINES="RSFM_BF_WAVES=4"
    return ["-D" + d for d in os.environ.get("RSFM_DEFINES", "").split() if d]


def _compile(src):
    path = os.path.join(CSRC, src)
    obj = os.path.join(OBJDIR, src + ".o")
    if src.endswith(".hip"):
        cmd = [HIPCC, "-x", "hip"] + COMMON + _defines() + DEVICE + ["-c", path, "-o", obj]
    else:
        cmd = [HIPCC] + COMMON + ["-c", path, "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    # the host pass does not know the packed-fp32 feature and says so; drop that line
    noise = "'-packed-fp32-ops' is not a recognized feature"
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l)
    if r.returncode != 0:
        raise RuntimeError("compile failed: %s\n%s" % (" ".join(cmd), err))
    if err.strip():
        sys.stderr.write(err + "\n")
    return obj


def build(verbose=False, out=None):
    """Compile and link; `out` overrides the library path (default in-tree)."""
    os.makedirs(OBJDIR, exist_ok=True)
    with ThreadPoolExecutor(max_workers=min(8, len(SOURCES))) as ex:
        objs = list(ex.map(_compile, SOURCES))
    lib = out or LIB
    tmp = lib + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", "--offload-arch=" + ARCH, "-o", tmp] + objs + ["-lamdhip64"]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed: %s\n%s" % (" ".join(cmd), r.stderr))
    os.replace(tmp, lib)
    if verbose:
        print("built", lib)
    if out is None:
        build_cpp_tests(verbose)
        build_hip_tests(verbose)
    return lib


def build_cpp_tests(verbose=False):
    """The C++ adapter test (tests/cpp/test_adapters): host code over
    include/rsfm_amd.hpp, linked against the in-tree library."""
    src = os.path.join(ROOT, "tests", "cpp", "test_adapters.cpp")
    if not os.path.exists(src):
        return None
    exe = os.path.join(ROOT, "tests", "cpp", "test_adapters")
    cmd = ["g++", "-O2", "-std=c++17", "-Wall", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include", "-I" + INCLUDE, src,
           "-L" + HERE, "-lrsfm_amd", "-L/opt/rocm/lib", "-lamdhip64", "-Wl,-rpath,$ORIGIN/../../rapidsfm_amd",
           "-Wl,-rpath,/opt/rocm/lib", "-o", exe]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("C++ adapter test failed to build: %s\n%s" % (" ".join(cmd), r.stderr))
    if verbose:
        print("built", exe)
    return exe


def build_hip_tests(verbose=False):
    """The GPU test's kernel for the matrix unit's sums (tests/hip/libmfma_sums.so)."""
    src = os.path.join(ROOT, "tests", "hip", "mfma_sums.hip")
    if not os.path.exists(src):
        return None
    lib = os.path.join(ROOT, "tests", "hip", "libmfma_sums.so")
    cmd = [HIPCC, "-x", "hip"] + COMMON + DEVICE + ["-shared", src, "-o", lib]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("GPU test kernel failed to build: %s\n%s" % (" ".join(cmd), r.stderr))
    if verbose:
        print("built", lib)
    return lib


if __name__ == "__main__":
    build(verbose=True)
