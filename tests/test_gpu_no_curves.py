"""Scenes without curves after a scene with many on the same handle: the path segments and counts of the frame
are all zero, and no path overflows its predicted capacity."""
from __future__ import annotations

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _points_only(n_paths):
    """Three points on the canvas per path, no curves."""
    path = np.repeat(np.arange(n_paths, dtype=np.uint32), 3)
    pos = np.random.default_rng(n_paths).uniform(10.0, 500.0, (3 * n_paths, 2)).astype(np.float32)
    none = np.zeros(0, np.uint32)
    return pos, path, none, none, none, np.zeros(n_paths, np.uint32), np.full(n_paths, 0xFF336699, np.uint32)


@pytest.mark.parametrize("mode", ["plain", "debug", "learned", "batch"])
@pytest.mark.parametrize("n_paths", [0, 1, 16])
def test_segments_without_curves_are_zero(spr, mode, n_paths):
    full = spr.Scene.generate(2, 1, 64, 512)
    r = spr.Rasterizer(512, 512, compose=1, debug=mode == "debug",
                       mode=spr.MODE_LEARNED if mode == "learned" else spr.MODE_PLAIN)
    if mode == "learned":
        params = np.zeros(5410, np.float32)
        params[-16:] = 1.0  # every path is predicted to have nothing
        r.mlp_set_params(params)
        r.learned_set_margin(0.0, 0)
    if mode == "batch":
        r.load_batch([full], [(512, 512)])
        r.render(readback=False)
        r.load_batch([spr.Scene.create(*_points_only(n_paths))], [(512, 512)])
    else:
        r.load_scene(full)
        r.render(readback=False)
        assert r.export("seg").max() > 0
        r.load_paths(*_points_only(n_paths))
    for _ in range(3):
        r.render(readback=False)
        seg, counts = r.export("seg"), r.export("path_counts")
        assert seg.shape == (n_paths + 1,) and not seg.any()
        assert counts.size == 2 * n_paths and not counts.any()
        st = r.stats()
        assert (st.n_intersections, st.n_cells, st.n_spans) == (0, 0, 0)
        if mode == "learned":
            assert st.n_overflow_paths == 0
        assert (r.export("image") == 255).all()
    r.close()
