"""The composite of one row of cells against the oracle, bit for bit: canvases at the edges of the chunk
widths, more paths on a row than its list holds (512) and than a listing step examines, opaque and
translucent paths mixed (an opaque path hides what lies under it), each compose mode and anti-aliased."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _quads(rng, n, w, h):
    """n four-sided paths across the canvas, some of them reaching out of it."""
    x0, x1 = rng.uniform(-20, w, n), rng.uniform(1, w + 20, n)
    y0, y1 = rng.uniform(-2, h / 2, n), rng.uniform(h / 2, h + 2, n)
    slant = rng.uniform(-5, 5, (n, 2))
    pts = np.stack([np.stack([x0, y0], 1), np.stack([x1, y0 + slant[:, 0]], 1),
                    np.stack([x1 + slant[:, 1], y1], 1), np.stack([x0, y1], 1), np.stack([x0, y0], 1)], 1)
    alpha = np.where(rng.random(n) < 0.1, 255, rng.integers(0, 255, n)).astype(np.uint32)
    fill = rng.integers(0, 1 << 24, n).astype(np.uint32) | (alpha << np.uint32(24))
    k = np.arange(n, dtype=np.uint32)
    return dict(pos=pts.reshape(-1, 2).astype(np.float32), pos_path=np.repeat(k, 5),
                curve_pos=(5 * k[:, None] + np.arange(4, dtype=np.uint32)).reshape(-1),
                curve_type=np.full(4 * n, 2, np.uint32), curve_path=np.repeat(k, 4),
                rule=(k % 2).astype(np.uint32), fill=fill, width=w, height=h)


@pytest.mark.parametrize("compose,aa", [(0, 0), (1, 0), (1, 16)])
@pytest.mark.parametrize("w,n", [(1, 3), (31, 257), (512, 40), (513, 600), (1024, 70), (1025, 1100), (2048, 300),
                                 (2049, 700), (4096, 65), (4097, 1300), (4200, 9000)])
def test_row_against_the_oracle(spr, orc, w, n, compose, aa):
    h = 5
    a = _quads(np.random.default_rng(w + n), n, w, h)
    f = orc.Frame(a, w, h, compose=compose, threads=4, aa=aa)
    r = spr.Rasterizer(w, h, compose=compose, aa=aa)
    r.load_paths(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")))
    for _ in range(2):
        img = r.render()
        assert np.array_equal(img, f.image())
    r.close()
