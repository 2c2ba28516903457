"""What is measured of this framework: the calls a painting program makes.

Each case is one pass through the public entry points, from the smallest call
(one dab of a brush) to a whole painting session on a 4096 x 4096 canvas, a
batch of canvases, a group of served requests and a gradient step.  Sizes
come from the repository's own configurations (painty_amd/workload.py) and
bench.

`exact` computes the same results in float64 with plain torch operations:
the imprint's visits pixel by pixel (pickup, deposit, snapshot ring), the
Kubelka-Munk composite, the lit render, and the texture brush with its
smudge.
"""
from __future__ import annotations

import ctypes as C
import itertools
import math

import numpy as np
import torch

from painty_amd import _lib
from painty_amd import diff as D
from painty_amd import hip as H
from painty_amd import serve as SV
from painty_amd import workload as W

DEV = "cuda"


# ------------------------------------------------------------------ cases --
def listed():
    return [
        # one dab of a small brush on a window-sized canvas: a mouse press
        dict(name="dab", kind="dab", rows=480, cols=640, radius=8.0, snapshot=True),
        # one mouse move: a short spline painted with paintStroke, then the
        # canvas composed for display
        dict(name="mouse-stroke", kind="mouse", rows=600, cols=800, radius=20.0, points=5,
             step=12, snapshot=True),
        # a stroke list on one canvas (the 1024 x 1024, 200-stamp configuration)
        dict(name="list-1024", kind="list", rows=1024, cols=1024, radius=32.0, stamps=200,
             pickup=True, snapshot=True, clock=False),
        # a painting session in one call: strokes of different brushes, dried
        # every 500 stamps, then composed (the 4096 x 4096 configuration)
        dict(name="session-4096", kind="session", rows=4096, cols=4096, stamps=2000, fmin=129,
             fmax=257, dry_every=500),
        # composite of a large resident canvas
        dict(name="compose-4096", kind="compose", rows=4096, cols=4096, layers=1),
        # dry layer and wet layer over a substrate, odd size
        dict(name="compose2-767x1023", kind="compose", rows=767, cols=1023, layers=2),
        # the display path of a full-HD window: lit render, then 8-bit sRGB
        dict(name="display-1080", kind="display", rows=1080, cols=1920, bits=8),
        # many canvases at once, stamps and composites
        dict(name="batch-32", kind="batch", canvases=32, smin=256, smax=2048, nmin=50, nmax=500,
             fmin=32, fmax=128),
        # a training step: composite + stamping, forward and backward
        dict(name="grad-2048", kind="grad", rows=2048, cols=2048, radius=32.0, stamps=500,
             paints=64, snapshot=True),
        # a small gradient step, odd size
        dict(name="grad-383x511", kind="grad", rows=383, cols=511, radius=12.0, stamps=60,
             paints=8, snapshot=True),
        # requests on many canvases arriving together at the server
        dict(name="serve-16", kind="serve", requests=16, smin=512, smax=2048, nmin=10, nmax=400,
             fmin=32, fmax=128),
        # a textured stroke with smudging (768 x 1024 canvas, radius 40)
        dict(name="texture-768x1024", kind="texture", rows=768, cols=1024, radius=40.0,
             smudge=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["dab", "mouse", "list", "list", "session", "compose", "display", "batch",
                       "grad", "serve", "texture"])
    if kind == "dab":
        return dict(kind=kind, rows=_log(rng, 200, 2048), cols=_log(rng, 200, 2048),
                    radius=float(_log(rng, 3, 64)), snapshot=rng.random() < 0.8)
    if kind == "mouse":
        return dict(kind=kind, rows=_log(rng, 300, 1500), cols=_log(rng, 300, 1500),
                    radius=rng.choice([1.0, 0.5]) * _log(rng, 6, 50), points=rng.randint(3, 8),
                    step=rng.randint(4, 20), snapshot=rng.random() < 0.8)
    if kind == "list":
        return dict(kind=kind, rows=_log(rng, 256, 2048), cols=_log(rng, 256, 2048),
                    radius=float(_log(rng, 5, 80)), stamps=_log(rng, 20, 500),
                    pickup=rng.random() < 0.75, snapshot=rng.random() < 0.8,
                    clock=rng.random() < 0.25)
    if kind == "session":
        fmin = _log(rng, 17, 129)
        return dict(kind=kind, rows=_log(rng, 512, 4096), cols=_log(rng, 512, 4096),
                    stamps=_log(rng, 100, 1500), fmin=fmin, fmax=min(257, fmin * 2),
                    dry_every=rng.choice([0, 200, 500]))
    if kind == "compose":
        return dict(kind=kind, rows=_log(rng, 128, 4096), cols=_log(rng, 128, 4096),
                    layers=rng.choice([1, 2]))
    if kind == "display":
        return dict(kind=kind, rows=_log(rng, 256, 2160), cols=_log(rng, 256, 3840),
                    bits=rng.choice([8, 16]))
    if kind == "batch":
        smin = _log(rng, 128, 512)
        return dict(kind=kind, canvases=rng.randint(4, 32), smin=smin, smax=smin * 4,
                    nmin=_log(rng, 10, 60), nmax=_log(rng, 61, 400), fmin=16,
                    fmax=_log(rng, 32, 128))
    if kind == "grad":
        return dict(kind=kind, rows=_log(rng, 200, 1500), cols=_log(rng, 200, 1500),
                    radius=float(_log(rng, 6, 48)), stamps=_log(rng, 20, 400),
                    paints=rng.randint(2, 64), snapshot=rng.random() < 0.75)
    if kind == "serve":
        return dict(kind=kind, requests=rng.randint(4, 16), smin=_log(rng, 256, 512),
                    smax=_log(rng, 600, 2048), nmin=10, nmax=_log(rng, 40, 400), fmin=16,
                    fmax=_log(rng, 32, 128))
    return dict(kind=kind, rows=_log(rng, 256, 1100), cols=_log(rng, 256, 1100),
                radius=float(_log(rng, 10, 50)), smudge=rng.random() < 0.8)


# ----------------------------------------------------------------- inputs --
class _Ptr:
    """A device address as an object torch can wrap without a copy; the
    tensor keeps it, and with it the memory's owner, alive."""

    def __init__(self, owner, ptr, shape, typestr):
        self.owner = owner
        self.__cuda_array_interface__ = dict(shape=tuple(shape), typestr=typestr,
                                             data=(int(ptr), False), version=2)


def _view(owner, ptr, shape, typestr="<f4"):
    return torch.as_tensor(_Ptr(owner, ptr, shape, typestr), device=DEV)


def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed) & 0x7FFFFFFF)


def _uniform(g, shape, lo, hi):
    return torch.rand(shape, generator=g, device=DEV, dtype=torch.float32) * (hi - lo) + lo


def _layer(g, rows, cols):
    """K, S (3, rows, cols) log-uniform, V uniform with 30% bare pixels."""
    K = torch.exp(_uniform(g, (3, rows, cols), math.log(0.01), math.log(10.0)))
    S = torch.exp(_uniform(g, (3, rows, cols), math.log(0.1), math.log(5.0)))
    V = _uniform(g, (rows, cols), 0.0, 0.5)
    V[_uniform(g, (rows, cols), 0.0, 1.0) < 0.3] = 0.0
    return K, S, V


def _substrate(g, rows, cols):
    return _uniform(g, (3, rows, cols), 0.7, 0.95)


class _CanvasViews:
    """A canvas' device planes as torch tensors."""

    def __init__(self, cv, rows, cols):
        L, R0, h = cv.device_planes()
        self.wet = L
        self.rgb = _lib.DevRgb((C.c_void_p * 3)(*R0))
        self.ks = [_view(cv, p, (rows, cols)) for p in L.ks]
        self.V = _view(cv, L.v, (rows, cols), "<f8")
        self.R0 = [_view(cv, p, (rows, cols)) for p in R0]
        self.h = _view(cv, h, (rows, cols))

    def fill(self, K, S, V, R0):
        for c in range(3):
            self.ks[c].copy_(K[c])
            self.ks[3 + c].copy_(S[c])
            self.R0[c].copy_(R0[c])
        self.V.copy_(V)

    def all(self):
        return dict(ks=self.ks, V=self.V, R0=self.R0, h=self.h)


def _canvas(rows, cols, g):
    cv = H.Canvas(rows, cols)
    H.default_context().synchronize()  # its planes are cleared before they are filled
    views = _CanvasViews(cv, rows, cols)
    K, S, V = _layer(g, rows, cols)
    views.fill(K, S, V, _substrate(g, rows, cols))
    torch.cuda.synchronize()  # filled on torch's stream, used on the library's
    return cv, views


def _foot(radius):
    w = 2 * math.ceil(radius) + 1
    return W.gaussian_core(w, w / 4.0)


def _paint(rs):
    return (np.exp(rs.uniform(math.log(0.01), math.log(10.0), 3)).astype(np.float32),
            np.exp(rs.uniform(math.log(0.1), math.log(5.0), 3)).astype(np.float32))


def _strokes(case, seed):
    return W.strokes(case["rows"], case["cols"], case["stamps"], seed, stamps_per_stroke=(20, 60))


def _session_inputs(case, seed):
    """[(radius, footprint, stamps)] of a session, and the whole stamp list."""
    st = W.strokes(case["rows"], case["cols"], case["stamps"], seed,
                   stamps_per_stroke=(50, 150), reach=0.08)
    if case["dry_every"]:
        st["flags"][case["dry_every"] - 1::case["dry_every"]] |= W.DRY_AFTER
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    out = []
    for b in range(int(st["brush"].max()) + 1):
        F = 2 * int(rs.randint(case["fmin"] // 2, case["fmax"] // 2 + 1)) + 1
        out.append(((F - 1) / 2.0, W.noisy_core(F, W.Stream(seed, 400 + b)),
                    st[st["brush"] == b]))
    return out


def _mouse_path(case, seed):
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    p = np.array([rs.uniform(0.2, 0.8) * case["cols"], rs.uniform(0.2, 0.8) * case["rows"]])
    a, path = rs.uniform(0, 2 * math.pi), []
    for _ in range(case["points"]):
        path.append(p.copy())
        a += rs.uniform(-0.5, 0.5)
        p = p + case["step"] * np.array([math.cos(a), math.sin(a)])
    return np.array(path), _paint(rs)


def _batch_inputs(case, seed):
    """[(rows, cols, radius, stamps)]: the sizes are the case's, the strokes the seed's."""
    rs = np.random.RandomState(case["canvases"] * 1000 + case["smin"])
    jobs = []
    for j in range(case["canvases"]):
        rows, cols = (int(x) for x in rs.randint(case["smin"], case["smax"] + 1, 2))
        n = int(rs.randint(case["nmin"], case["nmax"] + 1))
        r = float(max(1, int(rs.randint(case["fmin"], case["fmax"] + 1)) // 2))
        st = W.strokes(rows, cols, n, (seed * 64 + j) & 0x7FFFFFFF, stamps_per_stroke=(20, 80),
                       reach=0.15)
        jobs.append((rows, cols, r, st))
    return jobs


def _grad_inputs(case, seed):
    st = W.strokes(case["rows"], case["cols"], case["stamps"], seed, stamps_per_stroke=(20, 60),
                   reach=0.15)
    palK, palS = W.palette()
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    Wt = rs.dirichlet(np.ones(len(palK)), case["paints"])
    dips = np.flatnonzero(st["flags"] & W.DIP)
    paint_of = np.full(len(st), -1, np.int32)
    paint_of[dips] = rs.randint(0, case["paints"], len(dips))
    return st, palK, palS, Wt, paint_of


def _grad_tensors(case, seed):
    g = _gen(seed)
    K, S, V = _layer(g, case["rows"], case["cols"])
    R0 = _substrate(g, case["rows"], case["cols"])
    low = _uniform(g, (1, 3, 9, 9), 0.2, 0.9)
    target = torch.nn.functional.interpolate(low, size=(case["rows"], case["cols"]),
                                             mode="bilinear", align_corners=True)[0]
    return K, S, V, R0, target.contiguous()


def _serve_inputs(case, seed):
    """Requests whose canvases, sizes and counts are the case's, their strokes the seed's."""
    reqs = W.served_requests(case["requests"], case["requests"] * 1000 + case["smin"],
                             side=(case["smin"], case["smax"]),
                             stamps=(case["nmin"], case["nmax"]), foot=(case["fmin"], case["fmax"]))
    for i, q in enumerate(reqs):
        q.stamps = W.strokes(q.side, q.side, len(q.stamps), (seed * 64 + i) & 0x7FFFFFFF,
                             stamps_per_stroke=(20, 80), reach=0.15)
    return reqs


def _texture_inputs(case, seed):
    """A curved stroke across the canvas, and a bristled thickness map."""
    rs = np.random.RandomState(seed & 0x7FFFFFFF)
    rows, cols, r = case["rows"], case["cols"], case["radius"]
    n = 8
    x = np.linspace(1.5 * r, cols - 1.5 * r, n)
    y = rows / 2 + (rows / 2 - 1.6 * r) * 0.8 * np.sin(np.linspace(0, 4.0, n) + rs.uniform(0, 6))
    path = np.stack([x, y + rs.uniform(-4, 4, n)], 1)
    hairs = rs.uniform(0.2, 1.0, (64, 1)) * np.sin(np.linspace(0.05, math.pi - 0.05, 64))[:, None]
    thick = np.clip(hairs + 0.1 * rs.uniform(-1, 1, (64, 256)), 0.0, 1.0)
    return path, thick, tuple(np.asarray(p, np.float64) for p in _paint(rs))


def _plane(n):
    return (n + 63) // 64 * 64


# ---------------------------------------------------------------- prepare --
_server = None
_canvas_ids = itertools.count(1)


def _get_server():
    global _server
    if _server is None:  # a serving program runs one server per device
        _server = SV.Server(n_slots=16, hbm_budget_bytes=64 << 30)
    return _server


class _Session:
    """The server canvases of one group of clients, ended with it."""

    def __init__(self, server, ids):
        self.server, self.ids = server, ids

    def __del__(self):
        try:
            for i in self.ids:
                self.server.release_canvas(i)
        except Exception:
            pass


def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    rs = np.random.RandomState((seed + 77) & 0x7FFFFFFF)
    s = dict(case=case)
    if kind in ("dab", "mouse", "list", "session", "compose", "display", "texture"):
        rows, cols = case["rows"], case["cols"]
        s["cv"], s["views"] = _canvas(rows, cols, g)
    if kind == "dab":
        s["brush"] = H.FootprintBrush(case["radius"], _foot(case["radius"]))
        s["brush"].setUseSnapshotBuffer(case["snapshot"])
        s["brush"].dip(_paint(rs))
        s["at"] = ((rs.uniform(0.1, 0.9) * cols, rs.uniform(0.1, 0.9) * rows),
                   rs.uniform(0, 2 * math.pi))
    elif kind == "mouse":
        s["path"], paint = _mouse_path(case, seed)
        s["brush"] = H.FootprintBrush(case["radius"], _foot(case["radius"]))
        s["brush"].setUseSnapshotBuffer(case["snapshot"])
        s["brush"].dip(paint)
        s["out"] = torch.empty((3, rows, cols), device=DEV)
    elif kind == "list":
        s["brush"] = H.FootprintBrush(case["radius"], _foot(case["radius"]))
        s["brush"].setUseSnapshotBuffer(case["snapshot"])
        s["brush"].setPickupRate(0.9 if case["pickup"] else 0.0)
        s["stamps"] = H.stamps_to_c(_strokes(case, seed))
        if case["clock"]:  # a manual clock: paint dries 60 s after it was laid
            s["cv"].setClock(_lib.CLOCK_MANUAL)
            s["cv"].setDryingTime(60000)
            s["cv"].setTime(1000000)
            s["cv"].setTimeMap(np.zeros((rows, cols), np.int64))
            s["now"] = 1000000
    elif kind == "session":
        strokes = _session_inputs(case, seed)
        s["strokes"] = [(r, f, H.stamps_to_c(st)) for r, f, st in strokes]
        s["brush"] = H.FootprintBrush(strokes[0][0], strokes[0][1])
        s["out"] = torch.empty((3, rows, cols), device=DEV)
    elif kind == "compose":
        if case["layers"] == 2:
            s["cv2"], s["views2"] = _canvas(rows, cols, g)
        s["out"] = torch.empty((3, rows, cols), device=DEV)
    elif kind == "display":
        s["rgb"] = torch.empty((3, rows, cols), device=DEV)
        s["img"] = torch.empty((rows, cols, 3), device=DEV,
                               dtype=torch.uint8 if case["bits"] == 8 else torch.int16)
    elif kind == "batch":
        s["keep"], s["V"] = [], []
        jobs = _batch_inputs(case, seed)
        arr = (_lib.BatchJob * len(jobs))()
        # the composites in one buffer, planes 16-byte aligned
        s["out"] = torch.zeros(3 * sum(_plane(j[0] * j[1]) for j in jobs), device=DEV)
        at = 0
        for k, (rows, cols, r, st) in enumerate(jobs):
            cv, views = _canvas(rows, cols, g)
            br = H.FootprintBrush(r, _foot(r))
            br.updateSnapshot(cv)
            c_st = H.stamps_to_c(st)
            arr[k].canvas, arr[k].brush = cv.h.value, br.h.value
            arr[k].stamps, arr[k].n_stamps = C.cast(c_st, C.POINTER(_lib.PntStamp)), len(c_st)
            for c in range(3):
                arr[k].out[c] = s["out"][at:].data_ptr()
                at += _plane(rows * cols)
            s["keep"].append((cv, br, c_st))
            s["V"].append(views.V)
        s["jobs"] = arr
        H.batch_set_config(16, 32, 1, 1)  # as waves, what the tuner picks for such batches
    elif kind == "grad":
        st, palK, palS, Wt, paint_of = _grad_inputs(case, seed)
        K, S, V, R0, s["target"] = _grad_tensors(case, seed)
        s["brush"] = H.FootprintBrush(case["radius"], _foot(case["radius"]))
        s["brush"].setUseSnapshotBuffer(case["snapshot"])
        s["runner"] = D.GradRunner(case["rows"], case["cols"], s["brush"], st, paint_of, palK,
                                   palS, case["paints"])
        s["params"] = [t.requires_grad_() for t in
                       (K, S, V, R0, torch.from_numpy(Wt).to(DEV))]
    elif kind == "serve":
        server = _get_server()
        reqs = _serve_inputs(case, seed)
        base = {}
        for q in reqs:
            if q.canvas_id not in base:
                base[q.canvas_id] = next(_canvas_ids)
        s["server"] = server
        s["session"] = _Session(server, list(base.values()))
        s["reqs"] = [(base[q.canvas_id], q, H.stamps_to_c(q.stamps)) for q in reqs]
        s["sides"] = {base[q.canvas_id]: q.side for q in reqs}
    elif kind == "texture":
        path, thick, paint = _texture_inputs(case, seed)
        s["brush"] = H.TextureBrush(thick)
        s["brush"].enableSmudge(case["smudge"])
        s["brush"].setRadius(case["radius"])
        s["brush"].dip(paint)
        s["path"] = path
    if "brush" in s and "cv" in s and kind in ("dab", "mouse", "list", "session") and \
            case.get("snapshot", True):
        s["brush"].updateSnapshot(s["cv"])  # the canvas is the one the brush is painting on
    H.default_context().synchronize()
    torch.cuda.synchronize()
    return s


# -------------------------------------------------------------------- run --
def _rgb(t):
    return _lib.DevRgb((C.c_void_p * 3)(*[t[c].data_ptr() for c in range(3)]))


def _compose(views, out):
    _lib.call("pnt_dev_compose_wet", H.default_context().h, out[0].numel(), views.wet, views.rgb,
              _rgb(out), None)


def run(s):
    case, kind = s["case"], s["case"]["kind"]
    if kind == "dab":
        s["brush"].imprint(s["at"][0], s["at"][1], s["cv"])
        return s["views"].all()
    if kind == "mouse":
        s["brush"].paintStroke(s["path"], s["cv"])
        _compose(s["views"], s["out"])
        return dict(s["views"].all(), out=s["out"])
    if kind == "list":
        if case["clock"]:  # half a minute later than the last time
            s["now"] += 30000000
            s["cv"].setTime(s["now"])
        s["brush"].imprintStamps(s["stamps"], s["cv"], _lib.EXEC_FUSED)
        return s["views"].all()
    if kind == "session":
        s["brush"].imprintStrokes(s["strokes"], s["cv"], _lib.EXEC_FUSED)
        _compose(s["views"], s["out"])
        return dict(s["views"].all(), out=s["out"])
    if kind == "compose":
        if case["layers"] == 1:
            _compose(s["views"], s["out"])
        else:
            _lib.call("pnt_dev_compose2_wet", H.default_context().h, s["out"][0].numel(),
                      s["views"].wet, s["views2"].wet, s["views"].rgb, _rgb(s["out"]), None)
        return s["out"]
    if kind == "display":
        _lib.call("pnt_dev_render", s["cv"].h, _rgb(s["rgb"]))
        _lib.call("pnt_dev_encode", H.default_context().h, s["rgb"][0].numel(), _rgb(s["rgb"]), 1,
                  case["bits"], s["img"].data_ptr(), None)
        return dict(rgb=s["rgb"], img=s["img"])
    if kind == "batch":
        _lib.call("pnt_batch_run", H.default_context().h, s["jobs"], len(s["jobs"]),
                  _lib.BATCH_ONE_LAUNCH)
        return dict(out=s["out"], V=s["V"])
    if kind == "grad":
        R = D.PaintStamps.apply(*s["params"], s["runner"])
        loss = ((R - s["target"]) ** 2).sum()
        gK, gS, gV, gR0, gW = torch.autograd.grad(loss, s["params"])
        return dict(R=R.detach(), gK=gK, gS=gS, gV=gV, gR0=gR0, gW=gW)
    if kind == "serve":
        tickets = [s["server"].submit(cid, q.side, q.side, st, q.radius, q.footprint,
                                      background=q.background) for cid, q, st in s["reqs"]]
        for t in tickets:
            s["server"].wait(t)
        outs = {}
        for cid, side in s["sides"].items():  # where each client's picture lies on the device
            cvh, comp = C.c_void_p(), _lib.DevRgb()
            _lib.call("pnt_server_canvas", s["server"].h, cid, C.byref(cvh), C.byref(comp))
            outs["%08d" % len(outs)] = [_view(s["session"], p, (side, side)) for p in comp.p]
        return outs
    s["brush"].paintStroke(s["path"], s["cv"])
    return s["views"].all()


# ------------------------------------------------------------------- work --
# FP64 operations of one pickup + deposit (three blends of six channels).
VISIT_FLOPS = 100
# FP32 operations of one pixel's Kubelka-Munk evaluation (three channels).
KM_FLOPS = 150


def _stamp_work(rows, cols, r, n):
    """n stamps of radius r along strokes: the canvas and snapshot pixels
    they sweep read and written once, the pickup map and footprint once."""
    w = 2 * math.ceil(r) + 1
    swept = min(rows * cols, w * w + 2 * n * w)
    return dict(bytes=(64 + 40) * swept + 32 * w * w, flops=VISIT_FLOPS * n * w * w)


def work(case):
    kind = case["kind"]
    px = case.get("rows", 0) * case.get("cols", 0)
    if kind == "dab":
        return _stamp_work(case["rows"], case["cols"], case["radius"], 1)
    if kind == "mouse":
        w = _stamp_work(case["rows"], case["cols"], case["radius"],
                        (case["points"] - 1) * case["step"])
        return dict(bytes=w["bytes"] + 56 * px, flops=w["flops"] + KM_FLOPS * px)
    if kind == "list":
        return _stamp_work(case["rows"], case["cols"], case["radius"], case["stamps"])
    if kind == "session":
        w = _stamp_work(case["rows"], case["cols"], (case["fmin"] + case["fmax"]) / 4.0,
                        case["stamps"])
        dries = case["stamps"] // case["dry_every"] if case["dry_every"] else 0
        return dict(bytes=w["bytes"] + (56 + 96 * dries) * px,
                    flops=w["flops"] + (1 + dries) * KM_FLOPS * px)
    if kind == "compose":
        return dict(bytes=(24 + 32 * case["layers"]) * px, flops=KM_FLOPS * case["layers"] * px)
    if kind == "display":
        return dict(bytes=(44 + 12 + 12 + 3 * case["bits"] // 8) * px, flops=2 * KM_FLOPS * px)
    if kind in ("batch", "serve"):
        total = dict(bytes=0, flops=0)
        if kind == "batch":
            jobs = [(h, w, r, len(st), 56) for h, w, r, st in _batch_inputs(case, 0)]
        else:  # a request's snapshot and, on a new canvas, its first state are written too
            jobs = [(q.side, q.side, q.radius, len(q.stamps), 56 + 64)
                    for q in _serve_inputs(case, 0)]
        for rows, cols, r, n, per_px in jobs:
            w = _stamp_work(rows, cols, r, n)
            total["bytes"] += w["bytes"] + per_px * rows * cols
            total["flops"] += w["flops"] + KM_FLOPS * rows * cols
        return total
    if kind == "grad":
        w = _stamp_work(case["rows"], case["cols"], case["radius"], case["stamps"])
        return dict(bytes=3 * w["bytes"] + (56 + 28 + 12 + 52 + 40) * px,
                    flops=4 * w["flops"] + 3 * KM_FLOPS * px)
    r = case["radius"]
    steps = case["cols"] if case["smudge"] else 0
    return dict(bytes=(8 + 64) * 2 * r * case["cols"] + 2 * 56 * 4 * r * r,
                flops=steps * 4 * r * r * 150 + 2 * r * case["cols"] * 600)


# K, S and R0 are float32 and V float64 everywhere; an imprint's arithmetic is
# float64, so what differs is where K and S are rounded along a chain of
# visits: 2e-8 of the planes against `exact`, more in the few pixels a chain
# visits hundreds of times.  The composite's float32 evaluation is within 6e-8
# and the gradient's within 5e-7.
def tolerance(case):
    if case["kind"] == "compose":
        return dict(rel=3e-7, max=1e-5)
    if case["kind"] == "display":  # bytes: a value next to a rounding edge
        return dict(rel=6e-7, max=1e-3, differ=1e-4)
    if case["kind"] == "grad":
        return dict(rel=2e-6, max=1e-3)
    return dict(rel=4e-7, max=1e-4)


# ------------------------------------------------------------------ exact --
EPS = float(np.finfo(np.float64).eps) * 1e4
F64 = torch.float64


def _km(K, S, R0, d):
    """Kubelka-Munk reflectance of a layer K, S (3, ...) of thickness d over R0."""
    S = torch.where(S.abs() <= EPS, torch.full_like(S, 1e-11), S)
    B = torch.sqrt(torch.clamp(K * (K + 2.0 * S), min=0.0))  # S b
    thin = d.abs() < EPS
    x = B * torch.where(thin, torch.ones_like(d), d)
    E = torch.expm1(2.0 * torch.clamp(x, max=20.0))
    t = 2.0 * B / E
    AB = S + K + B
    num = S * (1.0 - R0) + R0 * (S * (K + B) / AB + t)
    den = S * (1.0 - R0) + K + B + t
    return torch.where(thin, R0, num / den)


def _round_away(x):
    t = torch.trunc(x)
    return t + torch.sign(x) * ((x - t).abs() >= 0.5)


class _Geo:
    """A brush geometry: the footprint centred in its square pickup map."""

    def __init__(self, radius, core):
        w = core.shape[0]
        self.radius, self.side = radius, int(math.ceil(math.sqrt(2.0) * w))
        pad = (self.side - w) // 2
        full = np.zeros((self.side, self.side))
        full[pad:pad + w, pad:pad + w] = core
        self.fp = torch.from_numpy(full.reshape(-1)).to(DEV)
        self.hr = (self.side - 1) // 2


def _chain_levels(ic, m):
    """Dependency level of each visit (reference order): one more than the
    highest of the earlier visits of its canvas pixel and of its map cell."""
    n = len(ic)

    def prev(key):
        o = np.argsort(key, kind="stable")
        p = np.full(n, -1, np.int64)
        same = key[o][1:] == key[o][:-1]
        p[o[1:][same]] = o[:-1][same]
        return p

    pa, pb = prev(ic), prev(m)
    has = np.flatnonzero((pa >= 0) | (pb >= 0))
    lev = np.zeros(n + 1, np.int64)
    lev[n] = -1  # no earlier visit
    a, b = np.where(pa < 0, n, pa)[has], np.where(pb < 0, n, pb)[has]
    while True:
        new = np.maximum(lev[a], lev[b]) + 1
        if np.array_equal(new, lev[has]):
            return lev[:n]
        lev[has] = new


def _visits(cx, cy, theta, geo, rows, cols, all_visits=False):
    """[(canvas pixels, map cells)] of an imprint, level by level."""
    c, s = math.cos(-theta), math.sin(-theta)
    k = torch.arange(-geo.hr, geo.hr + 1, device=DEV, dtype=F64)
    x, y = torch.trunc(k + cx).long(), torch.trunc(k + cy).long()
    mx = _round_away((k * c)[None, :] - (k * s)[:, None] + float(geo.hr)).long()
    my = _round_away((k * s)[None, :] + (k * c)[:, None] + float(geo.hr)).long()
    ok = ((x >= 0) & (x < cols))[None, :] & ((y >= 0) & (y < rows))[:, None]
    ok &= (mx >= 0) & (my >= 0) & (mx < geo.side) & (my < geo.side)
    m = my * geo.side + mx
    if not all_visits:
        ok &= geo.fp[torch.where(ok, m, torch.zeros_like(m))] > 0.0
    at = torch.nonzero(ok.reshape(-1))[:, 0]
    m = m.reshape(-1)[at]
    ic = (y[:, None] * cols + x[None, :]).reshape(-1)[at]
    n = int(at.numel())
    if n == 0:
        return []

    def twice(z):
        ks = np.arange(-geo.hr, geo.hr + 1, dtype=np.float64)
        return int(np.sum(np.trunc(ks + z) == 0)) > 1

    if twice(cx) or twice(cy):  # a fractional centre straddles column/row 0
        lev = _chain_levels(ic.cpu().numpy(), m.cpu().numpy())
        return [(ic[i], m[i]) for i in
                (torch.from_numpy(np.flatnonzero(lev == q)).to(DEV) for q in range(lev.max() + 1))]
    idx = torch.arange(n, device=DEV)
    first = torch.full((geo.side * geo.side,), n, device=DEV, dtype=torch.long)
    first.scatter_reduce_(0, m, idx, "amin")
    second = first[m] != idx
    return [(ic[~second], m[~second]), (ic[second], m[second])]


def _blend(va, a, vb, b):
    vt = va + vb
    big = vt > 0.001
    return torch.where(big, (va * a + vb * b) / torch.where(big, vt, torch.ones_like(vt)), a)


def _visit(P, Cv, X, fh, pr, dr, paint, alias):
    """One pickup and deposit of n visits: pickup cells P (7, n), canvas Cv
    (7, n), pickup source X (7, n); alias: the source is the canvas."""
    cap = 1.0
    vL = (pr * X[6]) * fh
    go = vL > 0.001
    ks = torch.where(go, _blend(P[6], P[:6], vL, X[:6]), P[:6])
    vP = torch.where(go, P[6] + vL, P[6])
    vX = torch.where(go, X[6] - vL, X[6])
    vC = vX if alias else Cv[6]
    free = torch.clamp(cap - vP, min=0.0)
    src = _blend(vP, ks, free, paint[:, None])
    vB = cap * fh
    cks = _blend(vB, src, vC, Cv[:6])
    Cn = torch.cat([cks, (vB + vC)[None]])
    Pn = torch.cat([ks, (vP - (dr * vP) * fh)[None]])
    return Pn, Cn, (None if alias else vX)


def _ring(cx, cy, geo, rows, cols):
    """The snapshot's allowed box and the window interior left out of it."""
    hr, r = geo.hr, geo.radius
    box = (max(int(cy - hr - r), 0), min(int(cy + hr + r), rows - 1),
           max(int(cx - hr - r), 0), min(int(cx + hr + r), cols - 1))
    win = (int(cy - hr), int(cy + hr), int(cx - hr), int(cx + hr))
    return box, win


class _Paint:
    """A canvas in float64: wet layer L (7, rows * cols), R0, h, time map."""

    def __init__(self, K, S, V, R0):
        self.rows, self.cols = V.shape
        self.L = torch.cat([K.to(F64), S.to(F64), V.to(F64)[None]]).reshape(7, -1)
        self.R0 = R0.to(F64).reshape(3, -1).clone()
        self.h = torch.zeros(self.rows * self.cols, device=DEV, dtype=F64)
        self.time = None
        self.new_brush()

    def new_brush(self):
        self.snap = None
        self.P = None

    def dry(self, i=slice(None)):
        self.h[i] += self.L[6, i]
        self.R0[:, i] = _km(self.L[:3, i], self.L[3:6, i], self.R0[:, i], self.L[6, i])
        self.L[:, i] = 0.0

    def compose(self):
        return _km(self.L[:3], self.L[3:6], self.R0, self.L[6]).reshape(3, self.rows, self.cols)

    def imprint(self, cx, cy, theta, geo, paint, pr=0.9, dr=0.05, snapshot=True, now=None,
                dry_ms=0):
        if self.P is None or self.P.shape[1] != geo.side ** 2:
            self.P = torch.zeros((7, geo.side ** 2), device=DEV, dtype=F64)
        if snapshot:
            if self.snap is None:
                self.snap = self.L.clone()
            (y0, y1, x0, x1), (ty, by, tx, bx) = _ring(cx, cy, geo, self.rows, self.cols)
            if y1 >= y0 and x1 >= x0:
                cv = self.L.view(7, self.rows, self.cols)[:, y0:y1 + 1, x0:x1 + 1]
                sn = self.snap.view(7, self.rows, self.cols)[:, y0:y1 + 1, x0:x1 + 1]
                a, b = max(ty + 1, y0) - y0, min(by - 1, y1) - y0 + 1
                p, q = max(tx + 1, x0) - x0, min(bx - 1, x1) - x0 + 1
                if b <= a or q <= p:
                    sn.copy_(cv)
                else:
                    keep = sn[:, a:b, p:q].clone()
                    sn.copy_(cv)
                    sn[:, a:b, p:q] = keep
        for ic, m in _visits(cx, cy, theta, geo, self.rows, self.cols, now is not None):
            if now is not None:  # paint older than the drying time dries first
                old = ic[(self.L[6, ic] > 0.001) & (now - self.time[ic] >= dry_ms)]
                old = torch.unique(old)
                if dry_ms > 0:
                    self.dry(old)
                self.time[ic] = now
                act = geo.fp[m] > 0.0
                ic, m = ic[act], m[act]
            X = self.snap[:, ic] if snapshot else self.L[:, ic]
            P, Cn, vX = _visit(self.P[:, m], self.L[:, ic], X, geo.fp[m], pr, dr, paint,
                               not snapshot)
            self.P[:, m] = P
            self.L[:, ic] = Cn
            if snapshot:
                self.snap[6, ic] = vX

    def stamps(self, st, geo, **kw):
        for q in st:
            if q["flags"] & W.DIP:
                self.paint = _paint64(q["K"], q["S"])
                self.P = None
            self.imprint(float(q["cx"]), float(q["cy"]), float(q["theta"]), geo, self.paint, **kw)
            if q["flags"] & W.DRY_AFTER:
                self.dry()

    def all(self):
        sh = (self.rows, self.cols)
        return dict(ks=[self.L[c].reshape(sh) for c in range(6)], V=self.L[6].reshape(sh),
                    R0=[self.R0[c].reshape(sh) for c in range(3)], h=self.h.reshape(sh))


def _paint64(K, S):
    return torch.from_numpy(np.concatenate([K, S]).astype(np.float64)).to(DEV)


def _paint_of(case, g):
    K, S, V = _layer(g, case["rows"], case["cols"])
    return _Paint(K, S, V, _substrate(g, case["rows"], case["cols"]))


def _catmull(p, t):
    """Catmull-Rom through p[1], p[2] (tau = 1/2): value and derivative."""
    tau, t2 = 0.5, t * t
    t3 = t2 * t
    b = (-tau * t + 2.0 * tau * t2 - tau * t3, 1.0 + (tau - 3.0) * t2 + (2.0 - tau) * t3,
         tau * t + (3.0 - 2.0 * tau) * t2 + (tau - 2.0) * t3, -tau * t2 + tau * t3)
    d = (tau * (-3.0 * t2 + 4.0 * t - 1.0), -t * (-2.0 * tau + 3.0 * (tau - 2.0) * t + 6.0),
         (t - 1.0) * (3.0 * (tau - 2.0) * t - tau), tau * t * (3.0 * t - 2.0))
    at = [p[0][k] * b[0] + p[1][k] * b[1] + p[2][k] * b[2] + p[3][k] * b[3] for k in (0, 1)]
    der = [p[0][k] * d[0] + p[1][k] * d[1] + p[2][k] * d[2] + p[3][k] * d[3] for k in (0, 1)]
    return at, der


def _exact_render(P):
    """The lit composite, (3, rows, cols)."""
    rows, cols = P.rows, P.cols
    Kd, V = P.compose(), P.L[6].reshape(rows, cols)

    def unit(v):
        z = (v * v).sum(0)
        return torch.where(z > 0.0, v / torch.sqrt(torch.where(z > 0.0, z, torch.ones_like(z))), v)

    def dot(a, b):
        return (a * b).sum(0)

    Vx = torch.cat([V[:, :1], V, V[:, -1:]], 1)
    Vy = torch.cat([V[:1], V, V[-1:]], 0)
    one, zero = torch.full_like(V, 2.0), torch.zeros_like(V)
    va = unit(torch.stack([one, zero, Vx[:, 2:] - Vx[:, :-2]]))
    vb = unit(torch.stack([zero, one, Vy[2:] - Vy[:-2]]))
    n = unit(torch.cross(va, vb, dim=0))
    n = torch.stack([n[0], n[1], -n[2]])
    px = torch.arange(cols, device=DEV, dtype=F64)[None, :].expand(rows, cols)
    py = torch.arange(rows, device=DEV, dtype=F64)[:, None].expand(rows, cols)
    pix = torch.stack([px, py, V])

    def at(x, y, z):
        return torch.tensor([x, y, z], device=DEV, dtype=F64)[:, None, None]

    ld = unit(at(-200.0, -1500.0, -2000.0) - pix)
    light = unit(ld)
    v = unit(at(cols / 2.0, rows / 2.0, -100.0) - pix)
    h = unit(v + light)
    NH, VH = dot(n, h).clamp(min=0.0), dot(v, h).clamp(min=0.0)
    NV, NL = dot(n, v).clamp(min=0.0), dot(n, light).clamp(min=0.0)
    m, s = 0.5, 0.2
    x2 = NH * NH
    A = 1.0 / (m * m + x2 * x2 * math.pi)
    Bk = torch.exp(-((1.0 - x2) / x2) / (m * m))
    G = torch.minimum(2.0 * NH * NV / VH, 2.0 * NH * NL / VH).clamp(max=1.0)
    lit = (NL > 0.0) & (NV > 0.0)
    spec = torch.where(lit, A * Bk * G / (NL * NV), torch.zeros_like(V))
    beta = 15.0 / (4.0 * math.pi * dot(ld, ld))
    return (beta * NL * ((1.0 - s) * Kd + s * spec) + Kd * 0.2 * Kd).clamp(0.0, 1.0)


def _exact_grad(case, seed):
    st, palK, palS, Wt, paint_of = _grad_inputs(case, seed)
    K, S, V, R0, target = _grad_tensors(case, seed)
    rows, cols = case["rows"], case["cols"]
    params = [t.to(F64).requires_grad_() for t in (K, S, V, R0, torch.from_numpy(Wt).to(DEV))]
    geo = _Geo(case["radius"], _foot(case["radius"]))
    pal = torch.from_numpy(np.concatenate([palK, palS], 1)).to(DEV)
    L = torch.cat([params[0], params[1], params[2][None]]).reshape(7, -1)
    alias = not case["snapshot"]
    X, P, paint = L, None, None
    for i, q in enumerate(st):
        if q["flags"] & W.DIP:
            w = params[4][int(paint_of[i])]
            ws = float(w.detach().sum())
            paint = (w if abs(ws - 1.0) < 10e-6 else w / w.sum()) @ pal
            P = torch.zeros((7, geo.side ** 2), device=DEV, dtype=F64)
        cx, cy = float(q["cx"]), float(q["cy"])
        if not alias:
            (y0, y1, x0, x1), (ty, by, tx, bx) = _ring(cx, cy, geo, rows, cols)
            if y1 >= y0 and x1 >= x0:
                mask = torch.zeros((rows, cols), device=DEV, dtype=torch.bool)
                mask[y0:y1 + 1, x0:x1 + 1] = True
                mask[max(ty + 1, 0):max(by, 0), max(tx + 1, 0):max(bx, 0)] = False
                at = torch.nonzero(mask.reshape(-1))[:, 0]
                X = X.index_copy(1, at, L[:, at])
        for ic, m in _visits(cx, cy, float(q["theta"]), geo, rows, cols):
            src = L[:, ic] if alias else X[:, ic]
            Pn, Cn, vX = _visit(P[:, m], L[:, ic], src, geo.fp[m], 0.9, 0.05, paint, alias)
            P = P.index_copy(1, m, Pn)
            L = L.index_copy(1, ic, Cn)
            if not alias:
                X = X.index_copy(1, ic, torch.cat([src[:6], vX[None]]))
    R = _km(L[:3], L[3:6], params[3].reshape(3, -1), L[6]).reshape(3, rows, cols)
    loss = ((R - target.to(F64)) ** 2).sum()
    g = torch.autograd.grad(loss, params)
    return dict(R=R.detach(), gK=g[0], gS=g[1], gV=g[2], gR0=g[3], gW=g[4])


def _reflect(i, n):
    i = torch.where(i < 0, -i - 1, i)
    return torch.where(i >= n, 2 * n - i - 1, i).clamp(0, n - 1)


def _bilinear(img, x, y):
    """img (..., rows, cols) at (x, y), reflected borders."""
    rows, cols = img.shape[-2:]
    xi, yi = torch.floor(x), torch.floor(y)
    a, c = x - xi, y - yi
    xi, yi = xi.long(), yi.long()
    x0, x1 = _reflect(xi, cols), _reflect(xi + 1, cols)
    y0, y1 = _reflect(yi, rows), _reflect(yi + 1, rows)
    return (img[..., y0, x0] * (1.0 - a) + img[..., y0, x1] * a) * (1.0 - c) + \
        (img[..., y1, x0] * (1.0 - a) + img[..., y1, x1] * a) * c


def _spline_at(v, u):
    n = len(v)
    x = (n - 1) * u
    i = int(x)
    return _catmull([v[min(max(i - 1 + q, 0), n - 1)] for q in range(4)], x - math.floor(x))


def _unit2(t):
    z = t[0] * t[0] + t[1] * t[1]
    return [t[0] / math.sqrt(z), t[1] / math.sqrt(z)] if z > 0.0 else list(t)


def _mean_value(poly, val, px, py):
    """Mean value coordinates: values `val` at polygon `poly`, at points (px, py)."""
    sx, sy = poly[:, 0, None] - px[None], poly[:, 1, None] - py[None]
    r = torch.sqrt(sx * sx + sy * sy)
    nx, ny, nr = sx.roll(-1, 0), sy.roll(-1, 0), r.roll(-1, 0)
    A = (sx * ny - nx * sy) / 2.0
    Dt = sx * nx + sy * ny
    Ap, Dp, rp = A.roll(1, 0), Dt.roll(1, 0), r.roll(1, 0)
    w = torch.where(Ap != 0.0, (rp - Dp / r) / Ap, torch.zeros_like(A)) + \
        torch.where(A != 0.0, (nr - Dt / r) / A, torch.zeros_like(A))
    Wt = w.sum(0)
    return (w * val[:, 0, None]).sum(0) / Wt, (w * val[:, 1, None]).sum(0) / Wt


def _exact_texture(case, seed):
    path, thick, paint = _texture_inputs(case, seed)
    P = _paint_of(case, _gen(seed))
    rows, cols, r = P.rows, P.cols, case["radius"]
    v = [tuple(p) for p in path]
    d0 = _unit2([v[1][0] - v[0][0], v[1][1] - v[0][1]])
    d1 = _unit2([v[-1][0] - v[-2][0], v[-1][1] - v[-2][1]])
    v = [(v[0][0] - d0[0] * r, v[0][1] - d0[1] * r)] + v + \
        [(v[-1][0] + d1[0] * r, v[-1][1] + d1[1] * r)]
    nv = len(v)
    lo = [max(min(p[k] for p in v) - r, 0.0) for k in (0, 1)]
    hi = [min(max(p[k] for p in v) + r, float((cols, rows)[k] - 1)) for k in (0, 1)]
    length = 0.0
    for a, b in zip(v[:-1], v[1:]):
        length += math.sqrt((b[0] - a[0]) ** 2 + (b[1] - a[1]) ** 2)
    right, left = [], []
    for i in range(nv):
        u = i / (nv - 1)
        c, t = _spline_at(v, u)
        t = _unit2(t)
        right.append(((c[0] + r * -t[1], c[1] + r * t[0]), (u, 1.0)))
        left.append(((c[0] - r * -t[1], c[1] - r * t[0]), (u, 0.0)))
    ring = right[::-1] + left
    poly = torch.tensor([q[0] for q in ring], device=DEV, dtype=F64)
    uv = torch.tensor([q[1] for q in ring], device=DEV, dtype=F64)
    x0, y0, x1, y1 = int(lo[0]), int(lo[1]), int(hi[0]), int(hi[1])
    xs = torch.arange(x0, x1 + 1, device=DEV)
    ys = torch.arange(y0, y1 + 1, device=DEV)
    gx = xs[None, :].expand(len(ys), len(xs)).reshape(-1)
    gy = ys[:, None].expand(len(ys), len(xs)).reshape(-1)
    u, w = _mean_value(poly, uv, gx.to(F64), gy.to(F64))
    T = torch.from_numpy(thick).to(DEV)
    inside = (u >= 0) & (u <= 1) & (w >= 0) & (w <= 1)
    vt = _bilinear(T, torch.where(inside, u, 0.5) * T.shape[1],
                   torch.where(inside, w, 0.5) * T.shape[0])
    vt = torch.where(inside & (vt > 0.0), vt, torch.zeros_like(vt)).reshape(len(ys), len(xs))
    trows, tcols = int(hi[1] - lo[1] + 1), int(hi[0] - lo[0] + 1)
    tmap = torch.zeros((trows, tcols), device=DEV, dtype=F64)
    tmap[:len(ys), :len(xs)] = vt[:trows, :tcols]
    maxd = float(tmap.max())
    if case["smudge"] and maxd > 0.0:
        _smudge(P, v, length, lo, tmap, maxd, int(2.0 * r))
    cov = torch.nonzero(tmap.reshape(-1) > 0.0)[:, 0]
    ic = (cov // tcols + y0) * cols + cov % tcols + x0
    vt, vc = tmap.reshape(-1)[cov], P.L[6, ic]
    pt = torch.from_numpy(np.concatenate(paint)).to(DEV)[:, None]
    P.L[:6, ic] = (vc * P.L[:6, ic] + vt * pt) / (vc + vt)
    P.L[6, ic] = torch.maximum(vt, vc)
    return P.all()


def _smudge(P, v, length, lo, tmap, maxd, n):
    """Paint traded between the canvas and a map that turns along the stroke."""
    rows, cols = P.rows, P.cols
    odd = n + 1 if n % 2 == 0 else n
    c0, rad = odd / 2.0, odd * 0.5
    M = torch.zeros((7, n, n), device=DEV, dtype=F64)
    k = torch.arange(n, device=DEV)
    mx, my = k[None, :].expand(n, n), k[:, None].expand(n, n)
    px, py = mx.to(F64) - c0, my.to(F64) - c0
    rot, u = 0.0, 0.0
    trows, tcols = tmap.shape
    while u <= 1.0:
        ctr, t = _spline_at(v, u)
        t = _unit2(t)
        theta = math.atan2(t[1], t[0])
        dth = theta - rot
        while dth <= -0.5 * math.pi:
            dth += math.pi
        while dth > 0.5 * math.pi:
            dth -= math.pi
        rot = theta
        sn, cs = math.sin(dth), math.cos(dth)
        rx, ry = px * cs - py * sn + c0, px * sn + py * cs + c0
        out = (rx < 0) | (ry < 0) | (rx >= n) | (ry >= n)
        M = torch.where(out, M, _bilinear(M, torch.where(out, 0.0, rx), torch.where(out, 0.0, ry)))
        x, y = mx + int(ctr[0] - n / 2.0), my + int(ctr[1] - n / 2.0)
        tx, ty = torch.trunc(x - lo[0]).long(), torch.trunc(y - lo[1]).long()
        ok = (x >= 0) & (y >= 0) & (x < cols) & (y < rows)
        ok &= (tx >= 0) & (ty >= 0) & (tx < tcols) & (ty < trows)
        dx, dy = ctr[0] - x.to(F64), ctr[1] - y.to(F64)
        ok &= ~(torch.sqrt(dx * dx + dy * dy) > rad)
        Dv = torch.where(ok, tmap[ty.clamp(0, trows - 1), tx.clamp(0, tcols - 1)], 0.0)
        at = torch.nonzero((Dv > 0.0).reshape(-1))[:, 0]
        ic = (y * cols + x).reshape(-1)[at]
        d, p, c = Dv.reshape(-1)[at], M.reshape(7, -1)[:, at], P.L[:, ic]
        cl, pl = c[6] * 0.1 * d / maxd, p[6] * 0.1 * d / maxd
        cr, pr = c[6] - cl, p[6] - pl
        cn, pn = cr + pl, pr + cl
        cgo, pgo = cn > 0.001, pn > 0.001
        safe_c, safe_p = torch.where(cgo, cn, 1.0), torch.where(pgo, pn, 1.0)
        Cn = torch.cat([(cr * c[:6] + pl * p[:6]) / safe_c, cn[None]])
        Pn = torch.cat([(pr * p[:6] + cl * c[:6]) / safe_p, pn[None]])
        P.L[:, ic] = torch.where(cgo, Cn, c)
        M.reshape(7, -1)[:, at] = torch.where(pgo, Pn, p)
        u += 1.0 / length


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    rs = np.random.RandomState((seed + 77) & 0x7FFFFFFF)
    if kind == "dab":
        P = _paint_of(case, g)
        paint = _paint64(*_paint(rs))
        at = (rs.uniform(0.1, 0.9) * P.cols, rs.uniform(0.1, 0.9) * P.rows)
        P.imprint(at[0], at[1], rs.uniform(0, 2 * math.pi),
                  _Geo(case["radius"], _foot(case["radius"])), paint, snapshot=case["snapshot"])
        return P.all()
    if kind == "mouse":
        P, (path, paint) = _paint_of(case, g), _mouse_path(case, seed)
        geo, n = _Geo(case["radius"], _foot(case["radius"])), len(path)
        paint = _paint64(*paint)
        for i in range(n - 1):
            q = [path[max(i - 1, 0)], path[i], path[i + 1], path[min(i + 2, n - 1)]]
            dist = math.sqrt((q[2][0] - q[1][0]) ** 2 + (q[2][1] - q[1][1]) ** 2)
            for k in range(1, int(dist) + 1):
                at, der = _catmull(q, k / dist)
                P.imprint(float(at[0]), float(at[1]), math.atan2(der[1], der[0]), geo, paint,
                          snapshot=case["snapshot"])
        return dict(P.all(), out=P.compose())
    if kind == "list":
        P = _paint_of(case, g)
        kw = {}
        if case["clock"]:  # milliseconds
            P.time = torch.zeros(P.rows * P.cols, device=DEV, dtype=torch.long)
            kw = dict(now=31000, dry_ms=60000)
        P.stamps(_strokes(case, seed), _Geo(case["radius"], _foot(case["radius"])),
                 pr=0.9 if case["pickup"] else 0.0, snapshot=case["snapshot"], **kw)
        return P.all()
    if kind == "session":
        P = _paint_of(case, g)
        last = None
        for r, foot, st in _session_inputs(case, seed):
            if last is None or abs(last - r) >= 0.5:
                geo, last = _Geo(r, foot), r
            P.stamps(st, geo)
        return dict(P.all(), out=P.compose())
    if kind == "compose":
        A = _paint_of(case, g)
        R = A.compose()
        if case["layers"] == 2:
            B = _paint_of(case, g)
            R = _km(B.L[:3], B.L[3:6], R.reshape(3, -1), B.L[6]).reshape(R.shape)
        return R
    if kind == "display":
        rgb = _exact_render(_paint_of(case, g))
        return dict(rgb=rgb, img=None)
    if kind == "batch":
        outs, vs = [], []
        for rows, cols, r, st in _batch_inputs(case, seed):
            P = _paint_of(dict(rows=rows, cols=cols), g)
            P.stamps(st, _Geo(r, _foot(r)))
            outs.append(torch.nn.functional.pad(P.compose().reshape(3, -1),
                                                (0, _plane(rows * cols) - rows * cols)).reshape(-1))
            vs.append(P.L[6].reshape(rows, cols))
        return dict(out=torch.cat(outs), V=vs)
    if kind == "grad":
        return _exact_grad(case, seed)
    if kind == "serve":
        canvases = {}
        for q in _serve_inputs(case, seed):
            if q.canvas_id not in canvases:
                z = torch.zeros((3, q.side, q.side), device=DEV, dtype=F64)
                bg = np.array(q.background, np.float32).astype(np.float64)
                canvases[q.canvas_id] = _Paint(
                    z, z, z[0], torch.from_numpy(bg).to(DEV)[:, None, None].expand_as(z))
            P = canvases[q.canvas_id]
            P.new_brush()
            P.stamps(q.stamps, _Geo(q.radius, q.footprint))
        return {"%08d" % i: list(P.compose()) for i, P in enumerate(canvases.values())}
    return _exact_texture(case, seed)
