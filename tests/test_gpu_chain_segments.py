"""Long chains cut into segments (frames of 2^23 intersections and more, k_chain_segments): every
crossing against the oracle, bit for bit, with chains at the lengths where the lanes per chain change
(255 | 256, 511 | 512, 1023 | 1024) and beyond, of cubics and quadratics in both directions, some of them
starting very slowly, where the segments' first guesses are off."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LENGTHS = (254, 255, 256, 257, 510, 511, 512, 513, 1022, 1023, 1024, 1025, 2047, 4000)


def test_long_chains_match_the_oracle(spr, orc):
    rng = np.random.default_rng(5)
    size = 8192
    pos, path, cpos, ctype, cpath = [], [], [], [], []
    total, i = 0, 0
    while total < (1 << 23) + (1 << 20):
        nx, ny = LENGTHS[i % len(LENGTHS)], LENGTHS[(i * 5 + 3) % len(LENGTHS)]
        d = np.array([2.0 * nx, 2.0 * ny])
        p0 = rng.uniform(0.0, size - d)
        s = np.sort(rng.uniform(0.0, 1.0, (2, 2)), axis=0)  # inner control points, monotone in both axes
        if i % 3 == 0:
            s = s**4  # nearly flat start
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
        total += 2 * (nx + ny)
        i += 1
    pos = np.array(pos, np.float32)
    a = dict(pos=pos, pos_path=np.array(path, np.uint32), curve_pos=np.array(cpos, np.uint32),
             curve_type=np.array(ctype, np.uint32), curve_path=np.array(cpath, np.uint32),
             rule=(np.arange(i) % 2).astype(np.uint32), fill=np.full(i, 0xFF336699, np.uint32), width=size, height=size)
    f = orc.Frame(a, size, size, threads=8)
    r = spr.Rasterizer(size, size, debug=True)
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
    r.render(readback=False)
    st = r.stats()
    assert st.n_intersections >= 1 << 23 and st.n_wave_chains > 1000
    g, o = r.export("inter"), f.get("inter")
    assert g.shape == o.shape
    bad = np.flatnonzero((g.reshape(-1, 2) != o.reshape(-1, 2)).any(1))
    assert bad.size == 0, (bad.size, bad[:4], g.reshape(-1, 2)[bad[:4]], o.reshape(-1, 2)[bad[:4]])
    r.close()
