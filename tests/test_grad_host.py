"""The host side of the gradient runner on a stand-in for the HIP runtime
(tests/cpp/grad_state.cpp, host_hip.hpp): what it keeps from one call to the
next, when an allocation fails, and on which stream it copies.  No device is
used."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
CPP = os.path.join(ROOT, "tests", "cpp")


@pytest.fixture(scope="module")
def program(tmp_path_factory):
    exe = str(tmp_path_factory.mktemp("grad_state") / "grad_state")
    lib = os.path.join(ROOT, "painty_amd")
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-rdynamic",
                    "-I" + os.path.join(ROOT, "include"), os.path.join(CPP, "grad_state.cpp"),
                    "-o", exe, "-L" + lib, "-lpainty_hip", "-Wl,-rpath," + lib,
                    "-Wl,-rpath,/opt/rocm/lib", "-Wl,-rpath-link,/opt/rocm/lib"], check=True,
                   timeout=300, capture_output=True)
    return exe


@pytest.mark.skipif(not shutil.which("g++"), reason="needs a C++ compiler")
@pytest.mark.parametrize("check", ["failures", "streams", "brush", "again", "no-tape"])
def test_runner_state(program, check):
    r = subprocess.run([program, check], capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    assert ": 0 failures" in r.stdout
