"""Frames solved by chains (2^23 intersections and more) with curves whose ends lie far outside the canvas, where the
count pass reserves entries that the write pass does not write: each of those still needs a bucket, since the
scatter takes what is there as an index."""
from __future__ import annotations

import numpy as np
import pytest
from test_gpu_big_pieces import _closed, _load

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("far", [2.1e9, 4.4e9, 1e12, 1e30])
def test_far_ends_among_many_chains(spr, orc, far):
    size = 1500
    rng = np.random.default_rng(7)
    mid = np.array([size / 2 + 0.3, size / 2 - 0.7])
    curves = []
    for dx, dy in ((1.0, 1.0), (1.0, 0.4), (-0.7, 1.0), (1e-9, 1.0), (1.0, -1e-9)):
        d = np.array([dx, dy]) * far
        curves += [[mid - d, mid - d / 3, mid + d / 3, mid + d], [mid + d, mid, mid - d],
                   [mid, mid + d * 1e-3, mid + d / 2, mid + d], [mid - d, mid + 1.0]]
    for _ in range(4200):  # 2,000 crossings and more each, out and back
        corner = rng.integers(0, 2, 2)
        p = np.where(corner, size - 1 - rng.uniform(0, 90, 2), rng.uniform(0, 90, 2))
        q = np.where(corner, rng.uniform(0, 90, 2), size - 1 - rng.uniform(0, 90, 2))
        s = np.sort(rng.uniform(0.1, 0.9, (2, 2)), axis=0)
        curves.append([p, p + (q - p) * s[0], p + (q - p) * s[1], q])
    a = _closed(curves)
    print(f"[far chains] {far}", flush=True)
    images = []
    for kw in (dict(debug=True), dict(), dict(debug=True)):
        r = spr.Rasterizer(size, size, **kw)
        _load(r, a)
        r.render(readback=False)
        assert r.stats().n_intersections >= 1 << 23
        images.append(r.export("image"))
        r.close()
    assert np.array_equal(images[0], images[1]) and np.array_equal(images[0], images[2])
    if far < 2.0**32:
        assert np.array_equal(images[0], orc.Frame(a, size, size, threads=8).image().reshape(-1))
