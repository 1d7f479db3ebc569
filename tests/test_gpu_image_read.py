"""rq_render_read_image: the image's values and PPM bytes, for sizes around the
words the device writes and around the size up to which an image is read
through pinned memory; either output alone gives the same bytes."""
import ctypes as C

import numpy as np
import pytest

import rq as _rq
from conftest import log

pytestmark = pytest.mark.gpu


def _read(ren, rgb, ppm):
    ptr = lambda a: a.ctypes.data_as(C.c_void_p) if a is not None else None  # noqa: E731
    ren.ctx._check(_rq.lib().rq_render_read_image(ren.ctx.h, ren.h, ptr(rgb), ptr(ppm)))


# 43690 pixels are 131070 values, 43691 are 131073: the line is at 131072
@pytest.mark.parametrize("w,h", [(1, 1), (2, 1), (3, 1), (5, 7), (64, 48), (43690, 1), (43691, 1),
                                 (320, 240)])
@pytest.mark.parametrize("spp", [1, 3])
def test_image_and_bytes(ctx, O, w, h, spp):
    log(f"image {w}x{h} spp {spp}")
    p = _rq.render_defaults()
    p.width, p.height, p.spp, p.camera = w, h, spp, _rq.CAMERA_PHILOX
    p.emission[0], p.surface[1], p.sky[2] = 1.7, -0.3, 1.5  # values past both ends of a byte
    s = ctx.upload_scene(_rq.icosphere(3, 2, center=(0, 0, -5)))
    b = ctx.build_lbvh(s, _rq.MORTON_SCENE_AABB)
    ren = _rq.Renderer(ctx, p)
    try:
        for _ in range(2):
            ren.frame(b)
            rgb, ppm = ren.image()
        samples = ren.samples()["rgb"]
        total = samples.reshape(-1, spp, 3)[:, 0].copy()
        for k in range(1, spp):
            total += samples.reshape(-1, spp, 3)[:, k]
        assert np.array_equal(rgb.view(np.uint32), total.reshape(-1).view(np.uint32))
        assert np.array_equal(ppm, O.resolve_ppm(samples, w * h, spp))
        one, other = np.full(3 * w * h + 1, 7, np.float32), np.full(3 * w * h + 1, 7, np.uint8)
        _read(ren, one, None)
        _read(ren, None, other)
        assert np.array_equal(one[:-1].view(np.uint32), rgb.view(np.uint32)) and one[-1] == 7
        assert np.array_equal(other[:-1], ppm) and other[-1] == 7
    finally:
        ren.close()
        ctx.release(b)
        ctx.release(s)
