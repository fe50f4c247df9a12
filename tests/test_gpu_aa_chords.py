"""Cells crossed by many edges of one path, anti-aliased: the sample masks at the chord counts where
k_cell_cover changes its form (3 | 4, 30 | 31, and 64 chords loaded at a time), and with more
chords in a workgroup's records than fit in LDS at once (1,280), bit for bit against the oracle, for both fill rules, with half of the points on multiples of 1/32 so that they meet
sample columns, sample rows and cell edges exactly."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CHORDS = {"edges": (1, 2, 3, 4, 5, 30, 31, 32, 63, 64, 65, 129), "rounds": (30, 7, 29) * 30}


@pytest.mark.parametrize("name", list(CHORDS))
def test_cells_of_many_chords(spr, orc, name):
    chords = CHORDS[name]
    rng = np.random.default_rng(len(chords))
    w, h = 67, 61
    pos, path, cpos, cpath, rule = [], [], [], [], []
    for i, n in enumerate(2 * chords):
        # n edges inside one cell, entered and left through a far point
        cx, cy = 2.0 * rng.integers(1, w // 2 - 6), 2.0 * rng.integers(3, h // 2 - 2)
        q = rng.uniform(0.0, 2.0, (n + 1, 2))
        q = np.where(rng.random((n + 1, 2)) < 0.5, np.round(q * 32.0) / 32.0, q)
        far = np.array([cx + 9.3, cy - 4.7])
        pts = np.vstack([far, q + (cx, cy), far]).astype(np.float32)
        cpos += list(range(len(pos), len(pos) + len(pts) - 1))
        cpath += [i] * (len(pts) - 1)
        pos += pts.tolist()
        path += [i] * len(pts)
        rule.append(int(i < len(chords)))
    n_paths = len(rule)
    fill = rng.integers(0, 1 << 24, n_paths).astype(np.uint32) | np.uint32(0xA0000000)
    a = dict(pos=np.array(pos, np.float32), pos_path=np.array(path, np.uint32), curve_pos=np.array(cpos, np.uint32),
             curve_type=np.full(len(cpos), 2, np.uint32), curve_path=np.array(cpath, np.uint32),
             rule=np.array(rule, np.uint32), fill=fill, width=w, height=h)
    f = orc.Frame(a, w, h, compose=1, threads=4, aa=16)
    r = spr.Rasterizer(w, h, compose=1, aa=16)
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
    img = r.render()
    cm, ref = r.export("coverage"), f.get("cmask")
    assert cm.shape == ref.shape
    assert np.array_equal(cm, ref), np.flatnonzero(cm != ref)[:8]
    assert np.array_equal(img, f.image())
    r.close()
