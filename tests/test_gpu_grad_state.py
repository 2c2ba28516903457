"""What a gradient runner may count on between its calls: a brush on another
context that stamps elsewhere between the forward and the backward, a brush
whose rates and footprint change in between, and a second backward of one
forward, the brush having stamped canvases of other sizes.  Every gradient against the FP64 oracle's, with the bound of test_gpu_grad.py."""
import numpy as np
import pytest

from painty_amd import diff as D
from painty_amd import hip as H
from tests.test_gpu_grad import check_grad, from_planes, oracle_gradient, to_planes
from tests.test_gpu_grad_tape import edge_case

pytestmark = pytest.mark.gpu


@pytest.fixture(params=["whole", "segments"])
def tape(request, monkeypatch):
    if request.param == "segments":
        monkeypatch.setenv("PAINTY_GRAD_TAPE_MB", "0")
    return request.param


def make(c, brush_ctx=None):
    rows, cols = c["V"].shape
    br = H.FootprintBrush(c["radius"], c["core"].astype(np.float32), brush_ctx)
    br.setPickupRate(c["rates"][0])
    br.setDepositionRate(c["rates"][1])
    br.setUseSnapshotBuffer(c["snapshot"])
    run = D.GradRunner(rows, cols, br, c["stamps"], c["paint_of"], c["palK"], c["palS"],
                       c["W"].shape[0], seg_len=7)
    run.forward(*[to_planes(c[k]) for k in ("K", "S", "V", "R0")], c["W"])
    return br, run


def check(tag, run, gR, ref):
    g = run.backward(to_planes(gR))
    check_grad(tag, {"K": from_planes(g[0]), "S": from_planes(g[1]), "V": from_planes(g[2]),
                     "R0": from_planes(g[3]), "W": g[4]}, ref)


def test_brush_of_another_context(hip, oracle, tape):
    c = edge_case(True)
    gR = np.random.default_rng(6).normal(size=c["R0"].shape)
    ref = oracle_gradient(oracle, c, gR)[1]
    other = H.Context(0)
    br, run = make(c, other)
    cv = H.Canvas(*c["V"].shape, other)
    st = c["stamps"].copy()
    st["cx"], st["cy"] = st["cy"] + 3.25, st["cx"] + 2.5  # another plan in the same buffers
    br.imprintStamps(st, cv)
    check("other/" + tape, run, gR, ref)


def test_brush_changed_after_the_forward(hip, oracle, tape):
    c = edge_case(True)
    gR = np.random.default_rng(8).normal(size=c["R0"].shape)
    ref = oracle_gradient(oracle, c, gR)[1]
    br, run = make(c)
    core = c["core"].astype(np.float32)
    br.setRadius(c["radius"] + 5, np.ones((2 * (int(np.ceil(c["radius"])) + 5) + 1,) * 2, np.float32))
    br.setRadius(c["radius"], np.ascontiguousarray(core[::-1] * np.float32(0.5)))
    br.setPickupRate(0.3)
    br.setDepositionRate(0.6)
    check("changed/" + tape, run, gR, ref)


def test_backward_again(hip, oracle, tape):
    c = edge_case(True)
    gR = np.random.default_rng(9).normal(size=c["R0"].shape)
    ref = oracle_gradient(oracle, c, gR)[1]
    br, run = make(c)
    for k, side in enumerate((None, 40, 130)):
        if side:
            br.imprintStamps(c["stamps"], H.Canvas(side, side + 3))
        check("again%d/%s" % (k, tape), run, gR, ref)
