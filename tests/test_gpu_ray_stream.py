"""The ray stream of a query launch: every ray is traced once and its result
written at its own index, whatever the number of rays, slices and waves.
Rays straight down on three known columns (a miss, triangle 0, triangle 1)
give the expected answer in closed form."""
import numpy as np
import pytest

from conftest import log

pytestmark = pytest.mark.gpu


def _scene(rq):
    x = np.float32([10, 11, 10, 20, 21, 20])
    y = np.float32([-0.5, -0.5, 1, -0.5, -0.5, 1])
    z = np.float32([-1, -1, -1, -2, -2, -2])
    return rq.MeshArrays(x, y, z, np.arange(6, dtype=np.uint32))


def _rays(n):
    k = np.arange(n) % 3
    one, zero = np.ones(n, np.float32), np.zeros(n, np.float32)
    return dict(ox=(10 * k + 0.125).astype(np.float32), oy=zero, oz=zero, dx=zero, dy=zero,
                dz=-one, tmin=zero, tmax=np.full(n, np.inf, np.float32)), k


# one ray, a part of a wave, the last launch whose first slices cover every
# ray and the first one that takes slices from the counters (6144 waves of one
# 64-ray slice on 256 CUs at six waves per SIMD), then sizes that leave the
# segments unequal shares of large and small slices.
@pytest.mark.parametrize("slice_rays", [64, 256, 1024])
@pytest.mark.parametrize("n", [1, 63, 393216, 393217, 400003, 524288 + 64 * 7 + 1, 1500007])
def test_every_ray_once(ctx, rq, n, slice_rays):
    log(f"ray stream n={n} slices of {slice_rays}")
    rays, k = _rays(n)
    prim = np.int32([-1, 0, 1])[k]
    t = np.float32([np.inf, 1, 2])[k]
    s = ctx.upload_scene(_scene(rq))
    b = ctx.build_lbvh(s, rq.MORTON_SCENE_AABB)
    d = rq.DeviceRays.from_host(ctx, rays)
    h = {"prim": rq.DeviceArray(ctx, 4 * n), "t": rq.DeviceArray(ctx, 4 * n)}
    occ = rq.DeviceArray(ctx, n)
    streams = [None, ctx.stream_create()]
    saved = ctx.trace_slice()
    ctx.trace_slice(slice_rays, slice_rays)
    try:
        # later launches start from the counters' values after earlier ones
        for rep, st in enumerate((streams[0], streams[1], streams[1])):
            h["prim"].fill(0x7F)
            occ.fill(0x7F)
            ctx.sync()
            ctx.closest_hit_dev(b, d, h, stream=st)
            ctx.any_hit_dev(b, d, occ, stream=st)
            ctx.sync(st)
            assert np.array_equal(h["prim"].download(np.int32, n), prim), rep
            assert np.array_equal(h["t"].download(np.float32, n), t), rep
            assert np.array_equal(occ.download(np.uint8, n), prim >= 0), rep
        assert ctx.device_errors() == 0
    finally:
        ctx.trace_slice(*saved)
        ctx.sync()
        ctx.stream_destroy(streams[1])
        d.free()
        occ.free()
        for a in h.values():
            a.free()
        ctx.release(b)
        ctx.release(s)
