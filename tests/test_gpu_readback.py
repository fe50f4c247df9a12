"""Image readback into pageable memory (chunks of 32 KiB in two pinned segments of 2 MiB) against the
device image, at the edges of chunks and segments, into an unaligned and into a pinned array, and of
a batch's documents."""
from __future__ import annotations

import ctypes as C

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


class _Image:
    def __init__(self, r, w, h):
        self.__cuda_array_interface__ = {"shape": (h, w, 4), "typestr": "|u1", "data": (r.image_device_ptr(), False),
                                         "version": 2}


def _device_image(r, w, h):
    r.synchronize()
    return torch.as_tensor(_Image(r, w, h), device="cuda").cpu().numpy()


@pytest.mark.parametrize("w,h", [(1, 1), (127, 64), (128, 64), (129, 64), (512, 1024), (513, 1024), (1024, 1024),
                                 (1023, 1025), (1500, 1100), (2048, 2100)])
def test_readback_is_the_device_image(spr, w, h):
    r = spr.Rasterizer(w, h, compose=1)
    for seed in (1, 2):  # the second frame reuses the segments
        r.load_scene(spr.Scene.generate(0, seed, 8, max(w, h, 16)))
        img = r.render()
        assert np.array_equal(img, _device_image(r, w, h))
    raw = np.zeros(4 * w * h + 8, np.uint8)  # guard bytes on both sides
    r._c(spr.lib().spr_render_frame(r._h, C.c_void_p(raw.ctypes.data + 3)))
    assert np.array_equal(raw[3:-5], img.reshape(-1)) and not raw[:3].any() and not raw[-5:].any()
    pinned = torch.zeros(4 * w * h, dtype=torch.uint8, pin_memory=True)
    r._c(spr.lib().spr_render_frame(r._h, C.c_void_p(pinned.data_ptr())))
    assert np.array_equal(pinned.numpy(), img.reshape(-1))
    r.close()


def test_batch_readback(spr):
    sizes = [(33, 17), (700, 900), (1, 3), (301, 77)]
    scenes = [spr.Scene.generate(0, 5 + d, 6, max(wh)) for d, wh in enumerate(sizes)]
    b = spr.Rasterizer(64, 64, compose=1)
    b.load_batch(scenes, sizes)
    b.render(readback=False)
    for d, (w, h) in enumerate(sizes):
        r = spr.Rasterizer(w, h, compose=1)
        r.load_scene(scenes[d])
        r.render(readback=False)
        assert np.array_equal(b.batch_image(d), _device_image(r, w, h)), d
        r.close()
    b.close()
