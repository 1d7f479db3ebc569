"""The ray counts where a default launch changes: up to 16 rays a wave while the chip's
8192 waves (256 compute units, eight waves per SIMD) hold them all, then full waves of 64
on their first slices, then slices from the counters. Every ray is traced once and its
result written at its own index, launch after launch."""
import numpy as np
import pytest

from conftest import log
from test_gpu_ray_stream import _rays, _scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [2 * 8192, 2 * 8192 + 1, 16 * 8192, 16 * 8192 + 1, 64 * 8192,
                               64 * 8192 + 1, 64 * 8192 + 63])
def test_every_ray_once_at_the_edges(ctx, rq, n):
    log(f"ray stream edge n={n}")
    rays, k = _rays(n)
    prim = np.int32([-1, 0, 1])[k]
    s = ctx.upload_scene(_scene(rq))
    b = ctx.build_lbvh(s, rq.MORTON_SCENE_AABB)
    d = rq.DeviceRays.from_host(ctx, rays)
    h = {"prim": rq.DeviceArray(ctx, 4 * n)}
    occ = rq.DeviceArray(ctx, n)
    try:
        for _ in range(3):
            h["prim"].fill(0x7F)
            occ.fill(0x7F)
            ctx.closest_hit_dev(b, d, h)
            ctx.any_hit_dev(b, d, occ)
            assert np.array_equal(h["prim"].download(np.int32, n), prim)
            assert np.array_equal(occ.download(np.uint8, n), prim >= 0)
        assert ctx.device_errors() == 0
    finally:
        d.free()
        occ.free()
        h["prim"].free()
        ctx.release(b)
        ctx.release(s)
