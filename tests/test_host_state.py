"""Host code of the library on a stand-in for the HIP runtime
(tests/cpp/host_hip.hpp): what the gradient runner keeps from one call to the
next, when an allocation fails, and on which stream it copies
(grad_state.cpp); what a brush holds for a long stroke and keeps past
an empty one (stroke_state.cpp).  No
device is used."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")


def build(out, name):
    exe = str(out / name)
    lib = os.path.join(ROOT, "painty_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-rdynamic",
                    "-I" + os.path.join(ROOT, "include"), os.path.join(CPP, name + ".cpp"),
                    "-o", exe, "-L" + lib, "-lpainty_hip", "-Wl,-rpath," + lib,
                    "-Wl,-rpath,/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib"], check=True,
                   timeout=300, capture_output=True)
    return exe


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    return build(tmp_path_factory.mktemp("grad_state"), "grad_state")


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a C++ compiler")
@pytest.mark.parametrize("check", ["failures", "streams", "brush", "again", "no-tape", "maps"])
def test_runner_state(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert ": 0 failures" in r.stdout


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a C++ compiler")
def test_what_a_stroke_leaves_with_the_brush(tmp_path):
    r = subprocess.run([build(tmp_path, "stroke_state")], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
