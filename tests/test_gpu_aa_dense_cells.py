"""Runs of neighbouring cells with more than 30 chords each, anti-aliased (k_cell_cover lists them per workgroup
and its waves take them in turn): every mask against the oracle, bit for bit, for one such cell, as many as
a workgroup has waves and one more, and as many as it has records and more, alone and among others."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _zigzags(cells, chords, others):
    """Paths that go up and down `chords` times in each of `cells` cells of two neighbouring rows, one per fill
    rule, and before, between and after them a few rectangles."""
    pos, path, cpos, cpath, rule = [], [], [], [], []

    def add(pts, r):
        cpos.extend(range(len(pos), len(pos) + len(pts) - 1))
        cpath.extend([len(rule)] * (len(pts) - 1))
        pos.extend(pts)
        path.extend([len(rule)] * len(pts))
        rule.append(r)

    for r in (0, 1):
        n = cells * chords
        xs = np.linspace(4.0, 4.0 + 2.0 * cells, n + 1)
        ys = np.where(np.arange(n + 1) % 2 == 0, 9.1, 10.9) + 0.03 * np.sin(np.arange(n + 1) * 0.7)
        for k in range(others):
            x, y = 3.3 + 7.0 * k, 5.7 + 0.9 * k
            add([(x, y), (x + 11.2, y + 1.0), (x + 10.0, y + 9.0), (x - 1.0, y + 8.0), (x, y)], r)
        add([*zip(xs, ys), (xs[-1], 14.3), (4.0, 14.9), (xs[0], ys[0])], r)
    n = len(rule)
    return dict(pos=np.array(pos, np.float32), pos_path=np.array(path, np.uint32), curve_pos=np.array(cpos, np.uint32),
                curve_type=np.full(len(cpos), 2, np.uint32), curve_path=np.array(cpath, np.uint32),
                rule=np.array(rule, np.uint32), fill=np.full(n, 0xA0336699, np.uint32) + np.arange(n, dtype=np.uint32))


@pytest.mark.parametrize("cells,chords,others", [(1, 40, 0), (4, 33, 0), (5, 31, 3), (60, 70, 0), (60, 64, 5),
                                                 (700, 36, 0), (700, 129, 9)])
def test_dense_cells_match_the_oracle(spr, orc, cells, chords, others):
    w, h = max(96, 2 * cells + 10), 40
    a = _zigzags(cells, chords, others)
    f = orc.Frame(a, w, h, compose=1, threads=4, aa=16)
    r = spr.Rasterizer(w, h, compose=1, aa=16)
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
    r.render(readback=False)
    cm, ref = r.export("coverage"), f.get("cmask")
    assert cm.shape == ref.shape
    assert np.array_equal(cm, ref), np.flatnonzero(cm != ref)[:8]
    assert np.array_equal(r.export("image"), f.image().reshape(-1))
    r.close()


def test_dense_cells_are_covered_side_by_side(spr):
    """1,000 neighbouring cells of some 200 chords: covering them takes less than sorting their entries does (three
    buckets, a workgroup each).  One workgroup taking all cells in turn took more than twice that."""
    a = _zigzags(500, 200, 0)
    ms = {}
    for name, kw in (("aa", dict(aa=16)), ("debug", dict(debug=True))):  # the same sort, without the cover
        r = spr.Rasterizer(1024, 40, compose=1, **kw)
        r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
        times = []
        for _ in range(8):
            r.render(readback=False)
            times.append(r.stats().frame_ms)
        ms[name] = min(times[2:])
        r.close()
    print(f"[dense cells] {ms}", flush=True)
    assert ms["aa"] < 2.0 * ms["debug"]
