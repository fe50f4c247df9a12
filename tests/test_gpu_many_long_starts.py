"""Many curves whose first part is on the canvas: frames with more than 256 chains with long starts take the chain
passes whatever their size, where chains of 256 crossings and more are solved by a wave each, or, above 2,048 of
them, by a lane each.  Every crossing against the oracle, bit for bit, and the other kinds of frames the same image."""
from __future__ import annotations

import numpy as np
import pytest
from test_gpu_big_pieces import _load

pytestmark = pytest.mark.gpu


def _starts(n, scale, size, kind, extra=0):
    """n unclosed curves from a corner of the canvas to `scale` canvases away, then `extra` short ones."""
    rng = np.random.default_rng(n)
    d = rng.uniform(0.6, 1.0, (n, 1, 2)) * scale * size
    s = np.sort(rng.uniform(0.15, 0.9, (n, 2, 2)), axis=1)
    p0 = rng.uniform(0.0, 0.01, (n, 1, 2)) * size
    m = 4 if kind == "cubic" else 3
    pts = np.concatenate([p0, p0 + d * s[:, : m - 2], p0 + d], axis=1)
    pts[1::2, :, 0] = size - pts[1::2, :, 0]
    pts[2::4, :, 1] = size - pts[2::4, :, 1]
    pts[3::4, :, 1] = size - pts[3::4, :, 1]
    pos = pts.reshape(-1, 2)
    ctype = np.full(n, {"cubic": 4, "quad": 3, "arc": 0x13}[kind], np.uint32)
    cpos, count = m * np.arange(n), np.full(n, m)
    if extra:
        e = rng.uniform(0.0, size, (extra, 4, 2))
        cpos = np.concatenate([cpos, len(pos) + 4 * np.arange(extra)])
        count = np.concatenate([count, np.full(extra, 4)])
        ctype = np.concatenate([ctype, np.full(extra, 4, np.uint32)])
        pos = np.concatenate([pos, e.reshape(-1, 2)])
    total = n + extra
    ids = np.arange(total, dtype=np.uint32)
    return dict(pos=pos.astype(np.float32), pos_path=np.repeat(ids, count), curve_pos=cpos.astype(np.uint32),
                curve_type=ctype, curve_path=ids, rule=ids % 2, fill=np.full(total, 0xC0336699, np.uint32) + ids,
                curve_weight=np.full(total, 0.7, np.float32) if kind == "arc" else None)


def _scene(spr, a):
    return spr.Scene.create(*(a[k] for k in ("pos", "pos_path", "curve_pos", "curve_type", "curve_path", "rule", "fill")),
                            curve_weight=a["curve_weight"])


# light chains; a wave each; a lane each; in the curve pass, a window with more long chains than waves take
@pytest.mark.parametrize("n,scale,size,kind,extra", [(700, 60, 400, "cubic", 0), (150, 40, 1600, "cubic", 0),
                                                     (150, 30, 1100, "quad", 0), (150, 30, 900, "arc", 0),
                                                     (1200, 60, 640, "cubic", 0), (120, 60, 142, "cubic", 4000)])
def test_many_long_starts_match_the_oracle(spr, orc, n, scale, size, kind, extra):
    a = _starts(n, scale, size, kind, extra)
    f = orc.Frame(a, size, size, threads=8)
    o = f.get("inter").reshape(-1, 2)
    assert len(o) < 1 << 23
    t = (o[:, 1] & ~3).view(np.float32)
    early = t < 1 / 32
    chains = np.bincount(2 * o[early, 0] + (o[early, 1] & 1))
    long_ = int((chains > 66).sum())
    print(f"[many long starts] {n} {kind} {size}: {len(o)} entries, {long_} long chains", flush=True)
    assert (long_ > 256) == (extra == 0)
    image = f.image().reshape(-1)
    r = spr.Rasterizer(size, size, debug=True)
    r.load_scene(_scene(spr, a))
    r.render(readback=False)
    g = r.export("inter").reshape(-1, 2)
    assert g.shape == o.shape
    bad = np.flatnonzero((g != o).any(1))
    assert bad.size == 0, (bad.size, bad[:4], g[bad[:4]], o[bad[:4]])
    assert np.array_equal(r.export("image"), image)
    st = r.stats()
    if extra == 0:  # the chain passes count their chains of 256 crossings and more
        assert st.n_wave_chains == int((np.bincount(2 * o[:, 0] + (o[:, 1] & 1)) >= 256).sum())
    r.close()
    r = spr.Rasterizer(size, size)
    r.load_scene(_scene(spr, a))
    for _ in range(2):
        r.render(readback=False)
        assert np.array_equal(r.export("image"), image)
    r.close()


def test_learned_frames_follow_what_they_saw(spr):
    """A learned frame takes the chain passes once the one before it had many long starts, and back; captured frames keep
    their route.  All of them the plain frame's image."""
    size = 400
    many, few = (_starts(n, 60, size, "cubic") for n in (700, 40))
    images = []
    for a in (many, few):
        r = spr.Rasterizer(size, size)
        _load(r, a)
        r.render(readback=False)
        images.append(r.export("image"))
        r.close()
    r = spr.Rasterizer(size, size, mode=spr.MODE_LEARNED)
    r.learned_train(spr.Scene.generate(2, 4, 64, 512), epochs=1, chunk_paths=64)
    for k in (0, 1, 0):
        _load(r, (many, few)[k])
        for _ in range(5):
            r.render(readback=False)
            assert np.array_equal(r.export("image"), images[k])
    # the same scene seen closer: from few long starts to many and back
    m = np.eye(4, dtype=np.float32)
    _load(r, many)
    plain = spr.Rasterizer(size, size)
    _load(plain, many)
    for zoom in (0.05, 1.0, 1.0, 1.0, 0.05, 0.05, 0.05):
        m[0, 0] = m[1, 1] = zoom
        r.set_mvp(m)
        plain.set_mvp(m)
        r.render(readback=False)
        plain.render(readback=False)
        assert np.array_equal(r.export("image"), plain.export("image")), zoom
    r.close()
    plain.close()
