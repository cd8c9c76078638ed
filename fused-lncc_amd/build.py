"""Build libfused_lncc_hip.so for gfx950 in-tree: one hipcc job per translation unit, then link; and
_step.so, the eager step as a torch extension (host code only), with the host compiler.

Usage: ``python fused-lncc_amd/build.py [--jobs N]``. Both land next to the Python package
(``fused-lncc_amd/fused_lncc/``), objects under ``fused-lncc_amd/_build/``.
"""
import argparse
import concurrent.futures as cf
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "fused_lncc", "libfused_lncc_hip.so")
ARCH = os.environ.get("FUSED_LNCC_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -packed-fp32-ops off: no v_pk_{add,mul,fma}_f32 anywhere. No fast-math: IEEE fp32 throughout.
CFLAGS = ["-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-Wall",
          "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
SOURCES = ["lncc_fused_h1.hip", "lncc_fused_h2.hip", "lncc_fused_h3.hip", "lncc_fused_h4.hip",
           "lncc_forward.hip", "lncc_small.hip", "lncc_aux.hip", "lncc_capi.hip"]


def _compile(src):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    cmd = [HIPCC] + CFLAGS + ["-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    msgs = [ln for ln in (r.stdout + r.stderr).splitlines() if "not a recognized feature" not in ln]
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n" + "\n".join(msgs))
    return obj


def _build_step():
    """_step.so (csrc/torch_step.cpp) against the installed torch's headers and libraries. The torch
    libraries are found where torch loaded them from when the module is imported."""
    import sysconfig
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    out = os.path.join(os.path.dirname(LIB), "_step.so")
    cmd = ([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__"]
           + [a for i in inc for a in ("-isystem", i)] + [os.path.join(CSRC, "torch_step.cpp"), "-o", out + ".tmp"]
           + ["-L" + os.path.join(root, "lib"), "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"])
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("building _step.so failed:\n" + r.stdout + r.stderr)
    os.replace(out + ".tmp", out)


def build(jobs=None, verbose=True):
    os.makedirs(BUILD, exist_ok=True)
    jobs = jobs or min(len(SOURCES) + 1, os.cpu_count() or 1)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        step = ex.submit(_build_step)
        objs = list(ex.map(_compile, SOURCES))
        step.result()
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    a = ap.parse_args()
    try:
        build(a.jobs)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
