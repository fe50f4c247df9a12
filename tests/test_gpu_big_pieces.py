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
