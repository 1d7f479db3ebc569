"""Many short rays over small trees: rays of a wave end at every visit, their results
are written together later, and trees of few primitives are walked without sharing.
Every ray has its own result, whatever the refill threshold, on both sides of the
sizes where launches change; rays with an empty interval among them."""
import numpy as np
import pytest

import rq as _rq
from conftest import log
from helpers import random_soup

pytestmark = pytest.mark.gpu


def _rays(n, seed):
    g = np.random.default_rng(seed)
    p = g.uniform(-1.3, 1.3, (n, 3))
    o = np.zeros((n, 3)) + [0.0, 0.0, 5.0]
    d = (p - o) / np.linalg.norm(p - o, axis=1, keepdims=True)
    d = d.astype(np.float32)
    r = dict(ox=o[:, 0], oy=o[:, 1], oz=o[:, 2], dx=d[:, 0], dy=d[:, 1], dz=d[:, 2],
             tmin=np.zeros(n), tmax=np.full(n, np.inf))
    r = {k: np.ascontiguousarray(v, np.float32) for k, v in r.items()}
    r["tmax"][::7] = 5.0
    r["tmin"][::11] = np.inf  # an empty interval
    return r


# the primitive counts where sharing starts; the ray counts where waves become full
@pytest.mark.parametrize("prims", [1, 2, 80, 511, 512, 513])
@pytest.mark.parametrize("rays", [131071, 131073, 200001])
def test_small_trees(ctx, O, prims, rays):
    mesh = random_soup(prims, 3, spread=1.0, size=0.3)
    r = _rays(rays, prims)
    log(f"small tree: {prims} triangles, {rays} rays")
    s = ctx.upload_scene(mesh)
    b = ctx.build_lbvh(s, _rq.MORTON_SCENE_AABB)
    d = _rq.DeviceRays.from_host(ctx, r)
    hits = {k: _rq.DeviceArray(ctx, 4 * rays) for k in ("prim", "t", "u", "v")}
    occ = _rq.DeviceArray(ctx, rays)
    saved = ctx.trace_config()
    try:
        ob = O.OracleBVH(mesh, 1)
        o, oa = ob.closest(r), ob.any(r)
        for refill in (64, 16, 1):
            ctx.trace_config(saved[0], saved[1], refill)
            for a in (*hits.values(), occ):
                a.fill(0x5A)
            ctx.closest_hit_dev(b, d, hits)
            ctx.any_hit_dev(b, d, occ)
            assert np.array_equal(hits["prim"].download(np.int32, rays), o["prim"]), refill
            for k in ("t", "u", "v"):
                assert np.array_equal(hits[k].download(np.uint32, rays), o[k].view(np.uint32)), k
            assert np.array_equal(occ.download(np.uint8, rays), oa["occ"]), refill
        assert ctx.device_errors() == 0
    finally:
        ctx.trace_config(*saved)
        d.free()
        for a in (*hits.values(), occ):
            a.free()
        ctx.release(b)
        ctx.release(s)
