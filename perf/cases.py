"""The measured cases: what programs have this rasteriser do, through its public entry points.

A case is one of five kinds of call:

- ``frame``: a resident scene is drawn again, and the image stays on the device (a compositor, a
  texture, an encoder behind it) or, with ``host``, comes back as an array;
- ``pan``: the same in learned mode under a new view every frame, as a viewer does;
- ``open``: a new document goes to a handle that is kept, is drawn once, and its image comes back;
- ``batch``: several documents of their own sizes in one frame, each image read back;
- ``scan``: the standalone exclusive scan of int32 values on the caller's stream.

Scenes come from the library's generators (0 scribbles, 1 glyphs, 2 illustration) or from the
drawings that the tests hold; the seed picks the generated scene, or the view of a drawing.  Every
output is bytes or whole numbers, so none has a value in 64 bits to be compared with.
"""
from __future__ import annotations

import math
from pathlib import Path

import numpy as np
import torch

import vkscanlinepr_amd as V

_DRAWINGS = Path(__file__).resolve().parent.parent / "tests" / "golden" / "rvg"
_FILES = ("car", "chord", "drops", "embrace", "reschart", "tiger")
_SIZES = {"car": (900, 600), "chord": (960, 960), "drops": (516, 576), "embrace": (538, 576),
          "reschart": (1133, 691), "tiger": (495, 510)}
# the documents of a batch, round-robin: generator, share of the paths, width and height in
# parts of the batch's size (thumbnails, cards, pages and posters beside each other)
_DOCS = ((0, 0.05, 0.5, 0.5), (1, 1.0, 1.0, 0.75), (2, 0.4, 0.76, 0.49), (0, 0.02, 0.3, 1.0),
         (2, 1.0, 1.0, 1.0), (1, 0.25, 0.25, 0.25), (2, 0.01, 0.13, 0.13), (1, 0.8, 0.63, 0.47))


def _frame(name, scene, paths, w, h, compose, aa=0, host=False):
    return {"name": name, "kind": "frame", "scene": scene, "paths": paths, "w": w, "h": h,
            "compose": compose, "aa": aa, "host": host}


def listed():
    return [
        # a small sketch, drawn and handed back as an array: the smallest whole call
        _frame("sketch_512", 0, 16, 512, 512, V.COMPOSE_OVERWRITE, host=True),
        # the 64-path scene: few curves, each crossing the whole canvas
        _frame("scribbles_1024", 0, 64, 1024, 1024, V.COMPOSE_SRC_OVER),
        # a page of text: very many very short curves
        _frame("page_2048", 1, 20000, 2048, 2048, V.COMPOSE_SRC_OVER),
        # text as it is shown on a screen: anti-aliased, and a canvas that no tile divides
        _frame("page_aa_1333", 1, 5000, 1333, 999, V.COMPOSE_SRC_OVER, aa=16),
        # the large illustration, the benchmark's frame
        _frame("illustration_4096", 2, 5000, 4096, 4096, V.COMPOSE_SRC_OVER),
        # the same anti-aliased, the heaviest single frame
        _frame("illustration_4096_aa", 2, 5000, 4096, 4096, V.COMPOSE_SRC_OVER, aa=16),
        # an interactive viewer: a screen-sized illustration whose view moves every frame
        {"name": "pan_1920", "kind": "pan", "scene": 2, "paths": 2000, "w": 1920, "h": 1080,
         "compose": V.COMPOSE_SRC_OVER},
        # a drawing with arcs, affine transforms and gradient paints, at twice its size
        {"name": "car_gradients", "kind": "frame", "file": "car", "zoom": 2.0, "w": 1800, "h": 1200,
         "compose": V.COMPOSE_SRC_OVER, "aa": 0, "host": False},
        # a drawing that is opened, drawn once and handed back (a thumbnailer, a converter)
        {"name": "open_tiger", "kind": "open", "file": "tiger", "zoom": 2.0, "w": 990, "h": 1020,
         "compose": V.COMPOSE_OVERWRITE},
        # a service that draws many documents of mixed sizes per frame
        {"name": "batch_16", "kind": "batch", "docs": 16, "paths": 600, "size": 1024,
         "compose": V.COMPOSE_SRC_OVER},
        # the scan on its own: the benchmark's length, and a short ragged one
        {"name": "scan_1e8", "kind": "scan", "n": 100_000_000},
        {"name": "scan_100003", "kind": "scan", "n": 100_003},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["frame"] * 6 + ["drawing"] * 2 + ["pan", "open", "batch", "scan"])
    compose = rng.choice([V.COMPOSE_OVERWRITE, V.COMPOSE_SRC_OVER])
    if kind == "scan":
        return {"kind": "scan", "n": _log_int(rng, 1000, 100_000_000)}
    if kind == "batch":
        return {"kind": "batch", "docs": rng.randint(4, 24), "paths": _log_int(rng, 50, 1000),
                "size": _log_int(rng, 300, 1200), "compose": compose}
    if kind == "drawing" or (kind == "open" and rng.random() < 0.5):
        f, zoom = rng.choice(_FILES), round(math.exp(rng.uniform(math.log(0.5), math.log(4.0))), 3)
        w, h = (max(1, int(x * zoom)) for x in _SIZES[f])
        if kind == "open":
            return {"kind": "open", "file": f, "zoom": zoom, "w": w, "h": h, "compose": compose}
        aa = 16 if compose == V.COMPOSE_SRC_OVER and rng.random() < 0.3 else 0
        return {"kind": "frame", "file": f, "zoom": zoom, "w": w, "h": h, "compose": compose,
                "aa": aa, "host": rng.random() < 0.2}
    scene = rng.randrange(3)
    w = _log_int(rng, 256, 2048 if scene == 0 else 4096)
    h = min(4096, max(200, int(w * rng.uniform(0.5, 1.5))))
    paths = _log_int(rng, *((8, 64), (100, 20000), (30, 5000))[scene])
    if kind == "pan":
        return {"kind": "pan", "scene": scene, "paths": paths, "w": w, "h": h, "compose": compose}
    if kind == "open":
        return {"kind": "open", "scene": scene, "paths": paths, "w": w, "h": h, "compose": compose}
    aa = 16 if compose == V.COMPOSE_SRC_OVER and rng.random() < 0.3 else 0
    c = _frame("", scene, paths, w, h, compose, aa, host=rng.random() < 0.2)
    del c["name"]
    return c


def _scene(case, seed):
    if "file" in case:
        return V.Scene.load_rvg(_DRAWINGS / (case["file"] + ".rvg"))
    return V.Scene.generate(case["scene"], seed, case["paths"], max(case["w"], case["h"]))


def _view(case, seed):
    """The drawing at its zoom, moved by up to 2% of the canvas; generated scenes as they are."""
    m = np.eye(4, dtype=np.float32)
    if "file" in case:
        rng = np.random.default_rng(seed)
        m[0, 0] = m[1, 1] = case["zoom"]
        m[0, 3], m[1, 3] = rng.uniform(-0.02, 0.02, 2) * (case["w"], case["h"])
    return m


def _documents(case, seed):
    scenes, canvases = [], []
    for d in range(case["docs"]):
        kind, share, fw, fh = _DOCS[d % len(_DOCS)]
        w, h = max(16, int(case["size"] * fw)), max(16, int(case["size"] * fh))
        n = max(1, int(case["paths"] * share))
        scenes.append(V.Scene.generate(kind, 1000 * (seed % 1_000_000) + d, min(n, 64) if kind == 0 else n,
                                       max(w, h)))
        canvases.append((w, h))
    return scenes, canvases


class _DeviceImage:
    """The handle's device image as an array that torch can alias; it keeps the handle."""

    def __init__(self, r):
        self.r = r
        self.__cuda_array_interface__ = {"shape": (r.height, r.width, 4), "typestr": "|u1",
                                         "data": (r.image_device_ptr(), False), "version": 2}


def prepare(case, seed):
    kind = case["kind"]
    if kind == "scan":
        g = torch.Generator(device="cuda").manual_seed(seed)
        # per-element counts, as a count pass leaves them: the total stays below 2^31
        x = torch.randint(0, 20, (case["n"],), dtype=torch.int32, device="cuda", generator=g)
        s = {"kind": kind, "r": V.Rasterizer(64, 64), "x": x, "n": case["n"],
             "out": torch.empty(case["n"] + 1, dtype=torch.int32, device="cuda"), "stream": torch.cuda.Stream()}
        torch.cuda.synchronize()
        return s
    if kind == "batch":
        scenes, canvases = _documents(case, seed)
        r = V.Rasterizer(64, 64, compose=case["compose"])
        r.load_batch(scenes, canvases)
        return {"kind": kind, "r": r, "docs": len(scenes)}
    scene = _scene(case, seed)
    mode = V.MODE_LEARNED if kind == "pan" else V.MODE_PLAIN
    r = V.Rasterizer(case["w"], case["h"], compose=case["compose"], mode=mode, aa=case.get("aa", 0))
    s = {"kind": kind, "r": r, "host": case.get("host", False), "scene": scene}
    if kind == "pan":
        # a viewer has its predictor trained; a short training stands for the file it would load
        r.learned_train(V.Scene.generate(case["scene"], 4, 1000 if case["scene"] else 64, 512), epochs=10,
                        chunk_paths=500)
        s["step"] = 0
    r.set_mvp(_view(case, seed))
    if kind != "open":
        r.load_scene(scene)
    if kind != "open" and not s["host"]:
        s["image"] = torch.as_tensor(_DeviceImage(r), device="cuda")
    return s


def run(state):
    kind, r = state["kind"], state["r"]
    if kind == "scan":
        r.scan_i32(state["x"].data_ptr(), state["out"].data_ptr(), state["n"], state["stream"].cuda_stream)
        return state["out"]
    if kind == "batch":
        r.render(readback=False)
        return [r.batch_image(d) for d in range(state["docs"])]
    if kind == "open":
        r.load_scene(state["scene"])
        return r.render()
    if kind == "pan":
        m = np.eye(4, dtype=np.float32)
        m[0, 3] = 2.0 * (state["step"] % 16 + 1)  # the view moves by two pixels a frame
        state["step"] += 1
        r.set_mvp(m)
    if state["host"]:
        return r.render()
    r.render(readback=False)
    return state["image"]


def _crossings(a, m, w, h):
    """About how many grid lines (every second pixel row and column) the curves cross on the canvas."""
    pos = a["pos"].astype(np.float64) @ m[:2, :2].T + m[:2, 3]
    n = 0.0
    kinds = a["curve_type"]
    for k, ctrl in ((V.CURVE_LINE, 2), (V.CURVE_QUAD, 3), (V.CURVE_ARC, 3), (V.CURVE_CUBIC, 4)):
        c = a["curve_pos"][kinds == k]
        if not len(c):
            continue
        p = pos[c[:, None] + np.arange(ctrl)]                                   # curves x points x 2
        t = np.linspace(0.0, 1.0, 9)
        b = np.stack([math.comb(ctrl - 1, i) * t**i * (1 - t) ** (ctrl - 1 - i) for i in range(ctrl)])
        q = np.clip(np.einsum("cpx,pt->ctx", p, b), 0.0, (w + 2, h + 2))
        n += np.abs(np.diff(q, axis=1)).sum() / 2
    return n


def work(case):
    """Bytes: the scene (or the values) read once, the image (or the sums) written once.  Flops: per
    crossing the 24 halvings that fix its parameter's bits (2 each) and two evaluations of the
    curve (18 each), the least that tells the last bracket; per scanned value one addition."""
    if case["kind"] == "scan":
        return {"bytes": 8 * case["n"] + 4, "flops": case["n"]}
    if case["kind"] == "batch":
        scenes, canvases = _documents(case, 1)
        docs = [(s.arrays(), np.eye(4), w, h) for s, (w, h) in zip(scenes, canvases)]
    else:
        docs = [(_scene(case, 1).arrays(), _view(case, 1).astype(np.float64), case["w"], case["h"])]
    size = flops = 0.0
    for a, m, w, h in docs:
        size += 12 * len(a["pos_path"]) + 12 * len(a["curve_type"]) + 8 * len(a["rule"]) + 4 * w * h
        flops += (24 * 2 + 2 * 18) * _crossings(a, m, w, h)
    return {"bytes": float(size), "flops": float(flops)}
