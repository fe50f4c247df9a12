"""Small frames where a chain's segments near t = 0 are predicted from candidate starts (k_curves): one cubic, whose
first window is a batch of its own, so that the test can count the segments that take candidates.  Every
crossing against the oracle, bit for bit."""
from __future__ import annotations

import numpy as np
import pytest
from test_gpu_big_pieces import _closed, _load

pytestmark = pytest.mark.gpu


def _candidates(chains, ctrl):
    """Segments and candidate starts of a batch of one cubic piece over t = 0..1, by the kernel's rules: chains =
    crossings per axis, ctrl = the inner control values as shares of the way."""
    before = lambda n, t: min(n, int(n * (3 * ctrl[0] * t * (1 - t) ** 2 + 3 * ctrl[1] * t * t * (1 - t) + t**3) + 2))
    length = max(4, -(-sum(chains) // 112))
    segments = walks = starts = 0
    for n in chains:
        head = max(length, before(n, 1 / 32)) if n > length + length // 2 else n
        if n - head < length // 2:
            head = n
        rest = -(-(n - head) // length)
        segments += 1 + rest
        first = [head + (n - head) * j // rest for j in range(rest)]
        want = sum(16 if i < before(n, 1 / 16) else 8 for i in first if i < before(n, 1 / 8))
        if 0 < want <= 384 - starts:
            starts += want
            walks += 1
    return segments, walks, starts


@pytest.mark.parametrize("nx,ny", [(400, 300), (500, 480), (40, 950), (0, 900)])
@pytest.mark.parametrize("ctrl,some", [((1 / 3, 2 / 3), True), ((0.9, 1.0), True), ((0.05, 0.3), True), ((0.0, 0.0), False)])
def test_candidate_starts_match_the_oracle(spr, orc, nx, ny, ctrl, some):
    w, h = max(64, 2 * nx + 16), max(64, 2 * ny + 16)
    p0, d = np.array([7.0, 7.0]), np.array([2.0 * nx + (0.5 if nx else 0.0), 2.0 * ny + (0.5 if ny else 0.0)])
    a = _closed([[p0, p0 + ctrl[0] * d, p0 + ctrl[1] * d, p0 + d]])
    segments, walks, starts = _candidates([n for n in (nx, ny) if n], ctrl)
    print(f"[candidates] {nx} {ny} {ctrl}: {segments} segments, {walks} walks, {starts} starts", flush=True)
    # the route: few windows, 8 entries a curve and more, one round of segments, chains with slow segments
    f = orc.Frame(a, w, h, threads=4)
    o = f.get("inter").reshape(-1, 2)
    assert 256 < np.bincount(o[:, 0])[0] <= 1024 and segments <= 256
    assert (walks > 0) == some
    for debug in (True, False):
        r = spr.Rasterizer(w, h, debug=debug)
        _load(r, a)
        r.render(readback=False)
        if debug:
            g = r.export("inter").reshape(-1, 2)
            bad = np.flatnonzero((g != o).any(1))
            assert bad.size == 0, (bad.size, bad[:4], g[bad[:4]], o[bad[:4]])
        assert np.array_equal(r.export("image"), f.image().reshape(-1))
        r.close()
