"""Monotone pieces of more than 1,024 entries in frames below 2^23 intersections (k_big_pieces: a workgroup each,
their chains cut into segments)."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _closed(curves):
    """One path per curve (its points), closed by a line."""
    pos, path, cpos, ctype = [], [], [], []
    for i, pts in enumerate(curves):
        cpos += [len(pos), len(pos) + len(pts) - 1]
        ctype += [len(pts), 2]
        pos += [*pts, pts[0]]
        path += [i] * (len(pts) + 1)
    n = len(curves)
    return dict(pos=np.array(pos, np.float32), pos_path=np.array(path, np.uint32), curve_pos=np.array(cpos, np.uint32),
                curve_type=np.array(ctype, np.uint32), curve_path=np.repeat(np.arange(n, dtype=np.uint32), 2),
                rule=(np.arange(n) % 2).astype(np.uint32), fill=np.full(n, 0xC0336699, np.uint32))


def _load(r, a):
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))


@pytest.mark.parametrize("w,h,nx,ny,cut", [(2048, 2048, 900, 1000, 2), (64, 4096, 0, 1800, 1), (64, 4096, 2, 1800, 1),
                                           (4096, 64, 1800, 0, 1), (4096, 64, 1800, 3, 1)])
def test_counts_the_chains_that_are_cut(spr, w, h, nx, ny, cut):
    """A cubic and the line back, of (nx, ny) crossings each at an even speed."""
    p0 = np.array([9.0, 9.0])
    d = np.array([2.0 * nx + (0.5 if nx else 0.0), 2.0 * ny + (0.5 if ny else 0.0)])
    r = spr.Rasterizer(w, h)
    _load(r, _closed([[p0 + d * t for t in (0.0, 1 / 3, 2 / 3, 1.0)]]))
    r.render(readback=False)
    st = r.stats()
    assert st.n_heavy_pieces == 2
    assert abs(st.n_intersections - 2 * (1 + nx + ny)) <= 4  # both pieces have their long axes
    assert st.n_wave_chains == 2 * cut
    r.close()


def _spans(k, n):
    """A cubic's, quadratic's or line's points from 0 to 1, by k: slow at its start, even, or slow at its end."""
    return {"slow": (0.0, 0.001, 0.02, 1.0), "even": (0.0, 1 / 3, 2 / 3, 1.0), "late": (0.0, 0.97, 0.999, 1.0),
            "quad": (0.0, 0.01, 1.0), "line": (0.0, 1.0)}[k][:n]


# pieces of 4,096 entries (the most that stay in LDS) and one more, and up to the longest of a canvas
@pytest.mark.parametrize("w,h,nx,ny", [(64, 16384, 0, 4095), (64, 16384, 0, 4096), (8192, 512, 3850, 245),
                                       (8192, 512, 3850, 246), (32, 16384, 9, 8180), (8192, 16, 4090, 5),
                                       (8192, 8192, 4000, 4080)])
@pytest.mark.parametrize("debug", [True, False])
def test_pieces_beyond_lds_match_the_oracle(spr, orc, w, h, nx, ny, debug):
    """Rising and falling curves of every type but arcs, slow and fast at their starts, each closed by a line."""
    p0 = np.array([3.0, 3.0])
    d = np.array([2.0 * nx + (0.5 if nx else 0.0), 2.0 * ny + (0.5 if ny else 0.0)])
    curves = []
    for k in ("slow", "even", "late", "quad", "line"):
        pts = [p0 + d * t for t in _spans(k, 4)]
        curves += [pts, pts[::-1], [np.array([w - q[0], q[1]]) for q in pts]]
    a = _closed(curves)
    print(f"[big-pieces] {w}x{h} {nx} {ny} debug={debug}", flush=True)
    f = orc.Frame(a, w, h, threads=8)
    o = f.get("inter").reshape(-1, 2)
    assert np.bincount(o[:, 0]).min() >= 1 + nx + ny - 4  # every curve is one long piece
    r = spr.Rasterizer(w, h, debug=debug)
    _load(r, a)
    r.render(readback=False)
    st = r.stats()
    assert st.n_heavy_pieces == len(a["curve_type"]) and st.n_intersections < 1 << 23
    assert st.n_intersections == len(o)
    if debug:
        g = r.export("inter").reshape(-1, 2)
        bad = np.flatnonzero((g != o).any(1))
        assert bad.size == 0, (bad.size, bad[:4], g[bad[:4]], o[bad[:4]])
    assert np.array_equal(r.export("image"), f.image().reshape(-1))
    r.close()


@pytest.mark.parametrize("far", [1e5, 5e8, 9.99e8, 1.01e9, 2.1e9, 4.4e9, 1e12, 1e30])
def test_far_ends_match_the_oracle(spr, orc, far):
    """Curves through the canvas whose ends lie far outside, where the count and the write pass round differently: the
    pieces that the count pass lists are those that the windows leave out.  Beyond 2^32 the count reserves
    entries that are not written, which the reference leaves undefined: there the two kinds of frame agree."""
    w = h = 3000
    mid = np.array([w / 2 + 0.3, h / 2 - 0.7])
    curves = []
    for dx, dy in ((1.0, 1.0), (1.0, 0.4), (-0.7, 1.0), (1e-9, 1.0), (1.0, -1e-9)):
        d = np.array([dx, dy]) * far
        curves += [[mid - d, mid - d / 3, mid + d / 3, mid + d], [mid + d, mid, mid - d],
                   [mid, mid + d * 1e-3, mid + d / 2, mid + d], [mid - d, mid + 1.0]]
    a = _closed(curves)
    print(f"[big-pieces] far {far}", flush=True)
    images = []
    for debug in (True, False):
        r = spr.Rasterizer(w, h, debug=debug)
        _load(r, a)
        r.render(readback=False)
        images.append(r.export("image"))
        if debug:
            g = r.export("inter")
        r.close()
    assert np.array_equal(images[0], images[1])
    if far < 2.0**32:
        f = orc.Frame(a, w, h, threads=8)
        assert np.array_equal(g, f.get("inter"))
        assert np.array_equal(images[0], f.image().reshape(-1))
