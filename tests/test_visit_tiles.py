"""The window tiles of the stamp kernels (visit_cell, tile_window, window_tile,
ring_scan in stampcore.hpp): the index arithmetic against the window walk on
the CPU (tests/cpp/cell_fuzz.cpp), and whole imprints where tiles, ring units
and their lists have edges, against the FP64 oracle."""
import os
import shutil
import subprocess

import numpy as np
import pytest

from painty_amd import workload as W
from tests.parity import compare_canvas, run_gpu, run_oracle

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
HIPCC = "/opt/rocm/bin/hipcc"


@pytest.mark.skipif(not shutil.which(HIPCC), reason="needs hipcc")
def test_visit_cells_match_the_window_walk(tmp_path):
    exe = str(tmp_path / "cell_fuzz")
    lib = os.path.join(ROOT, "painty_amd")
    subprocess.run([HIPCC, "--offload-arch=gfx950", "-std=c++17", "-O2",
                    "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(lib, "csrc"),
                    "-x", "hip", os.path.join(ROOT, "tests", "cpp", "cell_fuzz.cpp"), "-o", exe,
                    "-L" + lib, "-lpainty_hip", "-Wl,-rpath," + lib], check=True, timeout=600,
                   capture_output=True)
    r = subprocess.run([exe, "20000"], capture_output=True, text=True, timeout=600)
    assert r.returncode == 0, r.stdout + r.stderr
    assert ": 0 failures" in r.stdout


# radius 5: window of one tile; 11 and 23: footprint sides next to a multiple
# of 16; the canvas widths leave 0, 1 and 7 pixels past the last ring unit.
# A second stroke far from the first finds the ring dirty all over.
@pytest.mark.gpu
@pytest.mark.parametrize("radius", [1, 5, 11, 23])
@pytest.mark.parametrize("cols", [96, 97, 103])
@pytest.mark.parametrize("snapshot", [True, False])
def test_tile_and_ring_edges(hip, oracle, radius, cols, snapshot):
    wl = W.small(90, cols, 24, radius, 11 + radius, noisy=True)
    rs = np.random.RandomState(radius + cols)
    st = wl.stamps.copy()
    st["cx"][::5] = rs.uniform(-0.9 * radius, 0.0, len(st["cx"][::5]))  # across column 0
    st["cy"][1::7] = rs.uniform(-0.5, 0.5, len(st["cy"][1::7]))         # across row 0
    st["theta"][2::6] = np.pi / 4 * rs.randint(0, 8, len(st["theta"][2::6]))
    ocv, ob = run_oracle(wl, st, use_snapshot=snapshot)
    gcv, gb = run_gpu(wl, st, use_snapshot=snapshot, mode=2)
    compare_canvas("tiles/r%d/c%d/s%d" % (radius, cols, snapshot), gcv, ocv, pickup=(gb, ob))
