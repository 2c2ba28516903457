"""The two ways a differentiable list keeps what its adjoint needs -- the
whole list's visits on tape, or checkpoints and one segment's tape
(PAINTY_GRAD_TAPE_MB=0) -- against the FP64 oracle gradient, with the bound
of test_gpu_grad.py; a second backward of one forward; two runners on one
brush."""
import numpy as np
import pytest

from painty_amd import diff as D
from painty_amd import hip as H
from tests.test_gpu_grad import (check_grad, from_planes, gpu_run, oracle_gradient, to_planes)
from tests.test_oracle_grad import grad_case

pytestmark = pytest.mark.gpu


def edge_case(snapshot):
    """Strokes across canvas column/row 0 (shared-pixel levels), far ones, and
    a footprint side of one tile plus one."""
    c = grad_case(7, rows=70, cols=67, radius=8, n=24, snapshot=snapshot, n_paint=3)
    rs = np.random.RandomState(3)
    st = c["stamps"]
    st["cx"][::3] = rs.uniform(-7.0, 0.0, len(st["cx"][::3]))
    st["cy"][1::4] = rs.uniform(-0.6, 0.6, len(st["cy"][1::4]))
    return c


@pytest.mark.parametrize("snapshot", [True, False])
@pytest.mark.parametrize("tape", ["whole", "segments"])
def test_tape_and_checkpoints_match_oracle(hip, oracle, monkeypatch, tape, snapshot):
    if tape == "segments":
        monkeypatch.setenv("PAINTY_GRAD_TAPE_MB", "0")
    for name, c in (("edge", edge_case(snapshot)),
                    ("strokes", grad_case(13, rows=90, cols=101, radius=11, n=60, n_paint=5,
                                          reach=0.3, snapshot=snapshot))):
        gR = np.random.default_rng(2).normal(size=c["R0"].shape)
        _, g = gpu_run(c, gR, seg_len=7)
        _, ref = oracle_gradient(oracle, c, gR)
        check_grad("%s/%s/snap%d" % (name, tape, snapshot), g, ref)


def test_backward_twice_and_a_shared_brush(hip, oracle):
    c = edge_case(True)
    rows, cols = c["V"].shape
    br = H.FootprintBrush(c["radius"], c["core"].astype(np.float32))
    br.setPickupRate(c["rates"][0])
    br.setDepositionRate(c["rates"][1])

    def runner(stamps, paint_of):
        return D.GradRunner(rows, cols, br, stamps, paint_of, c["palK"], c["palS"],
                            c["W"].shape[0])

    ins = [to_planes(c[k]) for k in ("K", "S", "V", "R0")]
    gR = np.random.default_rng(4).normal(size=c["R0"].shape)
    a, b = runner(c["stamps"], c["paint_of"]), runner(c["stamps"][:9], c["paint_of"][:9])
    a.forward(*ins, c["W"])
    b.forward(*ins, c["W"])  # the same brush plans another list
    ref = oracle_gradient(oracle, c, gR)[1]
    for _ in range(2):
        g = a.backward(to_planes(gR))
        check_grad("again", {"K": from_planes(g[0]), "S": from_planes(g[1]),
                             "V": from_planes(g[2]), "R0": from_planes(g[3]), "W": g[4]}, ref)
