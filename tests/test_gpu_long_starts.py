"""Views of the first part of large curves: many crossings before t = 1 / 32, where guesses of a segment's start fail,
so that a wave solves the chain's first segment (k_curves, k_big_pieces).  Every crossing against the oracle, bit
for bit, for cubics in all directions and quadratics among them, as many long chains as a batch gives waves to
(8), more and fewer, and with pieces beyond a window."""
from __future__ import annotations

import numpy as np
import pytest
from test_gpu_big_pieces import _closed, _load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("curves,scale,size", [(1, 30, 1024), (4, 30, 400), (5, 20, 400), (6, 9, 1000), (40, 25, 500),
                                               (3, 40, 3000), (12, 12, 2300), (4200, 60, 142)])
def test_long_starts_match_the_oracle(spr, orc, curves, scale, size):
    """The curves start on the canvas and end `scale` canvases away, back to the start by a line.  Thousands of them
    have no lines: a window of 1,024 entries then holds more than 8 long chains."""
    rng = np.random.default_rng(curves * 100 + scale)
    parts = []
    for i in range(curves):
        d = rng.uniform(0.6, 1.0, 2) * scale * size
        s = np.sort(rng.uniform(0.15, 0.9, (2, 2)), axis=0)
        p0 = rng.uniform(0.0, 0.1 if curves < 1000 else 0.01, 2) * size
        quad = i % 5 == 3
        pts = [p0, *(p0 + d * s[k] for k in range(1 if quad else 2)), p0 + d]
        if i & 1:
            pts = [np.array([size - q[0], q[1]]) for q in pts]
        if i & 2:
            pts = [np.array([q[0], size - q[1]]) for q in pts]
        parts.append(pts)
    a = _closed(parts)
    if curves > 1000:
        keep = a["curve_type"] != 2
        a.update({k: a[k][keep] for k in ("curve_pos", "curve_type", "curve_path")})
    f = orc.Frame(a, size, size, threads=8)
    o = f.get("inter").reshape(-1, 2)
    # the chains (curve, axis) of cubics with more than 64 crossings before t = 1 / 32
    t = (o[:, 1] & ~3).view(np.float32)
    early = (t < 1 / 32) & (a["curve_type"][o[:, 0]] == 4)
    chains = np.bincount(2 * o[early, 0] + (o[early, 1] & 1))
    print(f"[long starts] {curves} {scale} {size}: {(chains > 64).sum()} long chains, "
          f"longest piece {np.bincount(o[:, 0]).max()}", flush=True)
    assert (chains > 64).sum() >= min(curves, 9)
    assert (np.bincount(o[:, 0]).max() > 1024) == (size > 2000)
    assert curves < 1000 or (len(o) >= 512 * 1024 and (chains > 64).sum() > 8.5 * len(o) / 1024)
    for debug in (True, False):
        r = spr.Rasterizer(size, size, debug=debug)
        _load(r, a)
        r.render(readback=False)
        if debug:
            g = r.export("inter").reshape(-1, 2)
            assert g.shape == o.shape
            bad = np.flatnonzero((g != o).any(1))
            assert bad.size == 0, (bad.size, bad[:4], g[bad[:4]], o[bad[:4]])
        assert np.array_equal(r.export("image"), f.image().reshape(-1))
        r.close()


def test_a_magnified_corner_is_no_slower_than_the_drawing(spr):
    """64 scribbles at 32 times their size have a sixteenth of the crossings on the canvas, most of them near t = 0.
    Correcting one guess after another there took 2.6 times the whole drawing's time."""
    r = spr.Rasterizer(1024, 1024, compose=1)
    r.load_scene(spr.Scene.generate(0, 1, 64, 1024))
    ms, n = [], []
    for zoom in (1.0, 32.0):
        m = np.eye(4, dtype=np.float32)
        m[0, 0] = m[1, 1] = zoom
        r.set_mvp(m)
        times = []
        for _ in range(12):
            r.render(readback=False)
            times.append(r.stats().frame_ms)
        ms.append(min(times[3:]))
        n.append(r.stats().n_intersections)
    print(f"[long starts] {n} crossings {ms} ms", flush=True)
    r.close()
    assert n[1] < n[0] / 10 and ms[1] < 2.0 * ms[0]
