"""Small frames whose curves start slowly, where the segments of a chain are predicted from candidate starts
(k_curves, frames of few windows): every crossing against the oracle, bit for bit, with one chain, as
many as the candidate list serves and more, and chains too short to be cut."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,lo,hi", [(1, 900, 1000), (3, 300, 1000), (20, 60, 700), (60, 2, 120), (200, 20, 900)])
def test_slow_starts_match_the_oracle(spr, orc, n, lo, hi):
    rng = np.random.default_rng(n)
    size = 1024
    pos, path, cpos, ctype, cpath = [], [], [], [], []
    for i in range(n):
        d = rng.uniform(lo, hi, 2)
        p0 = rng.uniform(0.0, size - d)
        s = np.sort(rng.uniform(0.0, 1.0, (2, 2)), axis=0) ** rng.integers(1, 6)
        quad = i % 4 == 1
        pts = [p0, *((p0 + d * s[k]) for k in range(1 if quad else 2)), p0 + d]
        if i & 1:
            pts = pts[::-1]
        if i & 2:
            pts = [np.array([size - q[0], q[1]]) for q in pts]
        cpos += [len(pos), len(pos) + len(pts) - 1]
        ctype += [3 if quad else 4, 2]
        cpath += [i, i]
        pos += [*pts, pts[0]]
        path += [i] * (len(pts) + 1)
    a = dict(pos=np.array(pos, np.float32), pos_path=np.array(path, np.uint32), curve_pos=np.array(cpos, np.uint32),
             curve_type=np.array(ctype, np.uint32), curve_path=np.array(cpath, np.uint32),
             rule=(np.arange(n) % 2).astype(np.uint32), fill=np.full(n, 0xFF336699, np.uint32), width=size, height=size)
    f = orc.Frame(a, size, size, threads=4)
    r = spr.Rasterizer(size, size, debug=True)
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
    img = r.render()
    g, o = r.export("inter"), f.get("inter")
    assert g.shape == o.shape and np.array_equal(g, o)
    assert np.array_equal(img, f.image())
    r.close()
