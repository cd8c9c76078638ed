"""The forward-only kernel's LDS accesses, checked on the host (tests/forward_lds_model.cpp) from the lane
maps, buffer offsets and step counts the kernel itself uses (fused-lncc_amd/csrc/lncc_geometry.h): bounds
and alignment, no float written twice or both written and read between two barriers, and every window of a
counted plane reading what was written for it, in a sequence of marches of odd and even lengths. Planted
mistakes (the roles on one buffer, an unclamped row, a march one step short, a neighbour's column, an odd
row offset) must be reported."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = os.path.join(ROOT, "tests", "forward_lds_model.cpp")
INC = os.path.join(ROOT, "fused-lncc_amd", "csrc")


@pytest.fixture(scope="module")
def model(tmp_path_factory):
    cxx = shutil.which("g++") or shutil.which("c++")
    if cxx is None:
        pytest.skip("no host C++ compiler")
    exe = str(tmp_path_factory.mktemp("flds") / "forward_lds_model")
    subprocess.run([cxx, "-std=c++17", "-O2", "-Wall", "-Werror", "-I", INC, SRC, "-o", exe], check=True)
    return exe


def test_forward_kernel_lds_accesses(model):
    r = subprocess.run([model], capture_output=True, text=True)
    assert r.returncode == 0, r.stdout + r.stderr
    lines = r.stdout.strip().splitlines()
    assert lines[-1] == "all ok" and len([ln for ln in lines if ln.endswith(": ok")]) == 7


@pytest.mark.parametrize("plant,kind", [(1, "written and read between two barriers"), (2, "a row past the input region"),
                                        (3, "planes counted"), (4, "not its window's"), (5, "reads at an odd float")])
def test_planted_mistakes_are_reported(model, plant, kind):
    r = subprocess.run([model, str(plant)], capture_output=True, text=True)
    assert r.returncode == 1 and kind in r.stdout, r.stdout
