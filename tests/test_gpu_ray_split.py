"""Rays walked by several lanes of a wave, and small launches spread over more
waves than their rays fill: whatever part of a tree each lane walks, the
closest hit is the lexicographic minimum (t, primitive) and any hit is whether
there is one, bit for bit as the oracle's."""
import numpy as np
import pytest

from conftest import log
from helpers import concat_rays, mesh_from, random_rays, random_soup, rays_toward

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _coplanar(n):
    """n triangles in one plane, the odd ones wound the other way: rays that
    start in the plane hit them at t = 0 and t = -0, which tie."""
    v = np.array([[-1, -1, -5], [1, -1, -5], [0, 1, -5]], np.float32)
    return mesh_from(np.concatenate([v[::-1] if k % 2 else v for k in range(n)]), np.arange(3 * n))


def _scene(kind):
    if kind == "overlap":  # every ray crosses most of the boxes: full stacks, deep ones
        return random_soup(3000, 17, spread=1.0, size=0.6), (
            rays_toward(40001, 43, target=(0, 0, 0), origin=(0.3, 0.2, 4)),
            random_rays(3000, 44, (-2, -2, -2), (2, 2, 2)))
    if kind == "ties":
        r = rays_toward(40001, 45)
        r["oz"] = r["oz"] - np.float32(5)
        r["tmin"] -= 1
        r["dz"][::3] = -1
        r["dx"][::3] = r["dy"][::3] = 0
        return _coplanar(301), (r,)
    # a few rays run along a row of slivers, through their boxes' corners and
    # past most of them; the other rays miss all
    g = np.random.default_rng(19)
    w = g.uniform(0.5, 1.0, (5000, 1, 1)) * np.array([[0, -1, -1], [0, 1, 1], [0, 1, 0.9]])
    m = mesh_from(w + np.linspace(0, 50, 5000)[:, None, None] * [1, 0, 0], np.arange(15000))
    r = rays_toward(40001, 46, target=(0, 30, 0), origin=(-1, 0.2, -0.2))
    long = slice(None, None, 61)
    jitter = g.uniform(-2e-2, 2e-2, (2, 40001)).astype(np.float32)
    r["dx"][long], r["dy"][long], r["dz"][long] = 1, jitter[0, long], jitter[1, long]
    return m, (r,)


# one wave, one ray in a block's second wave, rays for half the chip's waves
# at two a wave, the counts at which a wave gets four, and all of them
@pytest.mark.parametrize("kind", ["overlap", "ties", "row"])
@pytest.mark.parametrize("n", [1, 2, 3, 33, 64, 129, 4099, 16385, 40001])
def test_split_rays_match_oracle(ctx, O, rq, kind, n):
    mesh, parts = _scene(kind)
    rays = concat_rays(*parts)
    rays = {k: a[-n:].copy() if n <= 129 else a[:n].copy() for k, a in rays.items()}
    log(f"split rays {kind} n={n}")
    s = ctx.upload_scene(mesh)
    b = ctx.build_lbvh(s, 1)
    ob = O.OracleBVH(mesh, 1)
    o, oa = ob.closest(rays), ob.any(rays)
    saved = ctx.trace_config()
    try:
        for v in [v for v in ctx.trace_variants() if v["wide"]]:
            for refill in (16, 64):
                ctx.trace_config(v["index"], v["index"] if not v["tstack"] else 0, refill)
                g = ctx.closest_hit(b, rays)
                assert np.array_equal(g["prim"], o["prim"]), (v, refill)
                for k in ("t", "u", "v"):
                    assert np.array_equal(_bits(g[k]), _bits(o[k])), (k, v, refill)
                assert np.array_equal(ctx.any_hit(b, rays)["occ"], oa["occ"]), (v, refill)
        assert ctx.device_errors() == 0
    finally:
        ctx.trace_config(*saved)
        ctx.release(b)
        ctx.release(s)


# a serving step: tiles of 256 rays, the last one partial, walked to the end
@pytest.mark.parametrize("kind", ["overlap", "ties", "row"])
def test_split_rays_in_a_serving_step(ctx, O, rq, kind):
    mesh, parts = _scene(kind)
    rays = concat_rays(*parts)
    srv = rq.Server(0, mesh_slots=2, slot_tris=1 << 13, arena_bytes=64 << 20, max_inflight=8,
                    step_rays=1 << 16, chunk_rays=1 << 14, ray_tile=1024, hbm_budget=4 << 30)
    ob = O.OracleBVH(mesh, 1)
    try:
        slot = srv.load_mesh(mesh)
        jobs = []
        for n in (1, 255, 257, 4099, 40001):
            part = {k: a[-n:].copy() if n < 300 else a[:n].copy() for k, a in rays.items()}
            out = (np.empty(n, np.int32), np.empty(n, np.float32), np.empty(n, np.uint8))
            tk = srv.submit(n, rq.Q_CLOSEST | rq.Q_ANY, mesh=slot, rays=part, prim=out[0],
                            t=out[1], occ=out[2])
            jobs.append((part, out, tk))
        for part, out, tk in jobs:
            log(f"serving step {kind} n={len(out[0])}")
            srv.wait(tk)
            o = ob.closest(part)
            assert np.array_equal(out[0], o["prim"])
            assert np.array_equal(_bits(out[1]), _bits(o["t"]))
            assert np.array_equal(out[2], ob.any(part)["occ"])
    finally:
        srv.close()
