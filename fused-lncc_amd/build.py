"""Build libfused_lncc_hip.so for gfx950 in-tree: one hipcc job per translation unit, then link; and
_step, the eager step as a torch extension (host code only), with the host compiler.

Usage: ``python fused-lncc_amd/build.py [--jobs N] [--require-step]``. Both land next to the Python
package (``fused-lncc_amd/fused_lncc/``), objects under ``fused-lncc_amd/_build/``. The library needs
hipcc only. _step is optional (without it the Python autograd function does the same): where it
cannot be built, for want of torch, its headers or a host compiler, the reason goes to stderr and the
build succeeds; with ``--require-step`` it then fails, after the library is in place.
"""
import argparse
import concurrent.futures as cf
import os
import subprocess
import sys
import sysconfig

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "fused_lncc", "libfused_lncc_hip.so")
STEP = os.path.join(HERE, "fused_lncc", "_step" + sysconfig.get_config_var("EXT_SUFFIX"))   # for this interpreter
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
    """The extension (csrc/torch_step.cpp) against the installed torch's headers and libraries, which it
    names in itself. The torch libraries are found where torch loaded them from when it is imported."""
    import torch
    root = os.path.dirname(torch.__file__)
    inc = [os.path.join(root, "include"), os.path.join(root, "include", "torch", "csrc", "api", "include"),
           os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "include"), sysconfig.get_paths()["include"]]
    cmd = ([os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
            f'-DFL_TORCH="{torch.__version__} {torch.version.git_version}"', "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__"]
           + [a for i in inc for a in ("-isystem", i)] + [os.path.join(CSRC, "torch_step.cpp"), "-o", STEP + ".tmp"]
           + ["-L" + os.path.join(root, "lib"), "-ltorch", "-ltorch_cpu", "-ltorch_python", "-lc10", "-lc10_hip"])
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(r.stdout + r.stderr)
    os.replace(STEP + ".tmp", STEP)


def build(jobs=None, verbose=True, require_step=False):
    os.makedirs(BUILD, exist_ok=True)
    jobs = jobs or min(len(SOURCES) + 1, os.cpu_count() or 1)
    with cf.ThreadPoolExecutor(max_workers=jobs) as ex:
        step = ex.submit(_build_step)
        objs = list(ex.map(_compile, SOURCES))
    tmp = LIB + ".tmp"
    cmd = [HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", "-o", tmp] + objs
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    if verbose:
        print(f"built {LIB}")
    try:
        step.result()
    except Exception as e:   # a torch that does not load or is laid out otherwise, no compiler, a failed compilation
        if os.path.exists(STEP):   # of an earlier build
            os.remove(STEP)
        msg = f"building _step failed ({type(e).__name__}: {e})"
        if require_step:
            raise RuntimeError(msg) from e
        print(f"{msg}\nThe library is built; without _step the Python autograd function is used.", file=sys.stderr)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--jobs", type=int, default=None)
    ap.add_argument("--require-step", action="store_true", help="fail where _step cannot be built")
    a = ap.parse_args()
    try:
        build(a.jobs, require_step=a.require_step)
    except RuntimeError as e:
        print(e, file=sys.stderr)
        sys.exit(1)
