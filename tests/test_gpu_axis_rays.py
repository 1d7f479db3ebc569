"""Rays along the axes, or nearly, in scenes of every scale: 1/d is infinite or
huge there, and the distances to the planes of a wide node's grid must stay
ordered however large the grid's steps are. Closest and any hits of the wide
walks equal the oracle's bit for bit."""
import numpy as np
import pytest

import rq as _rq
from conftest import log
from helpers import concat_rays, random_soup

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _pack(o, d):
    o, d = np.asarray(o).astype(np.float32), np.asarray(d).astype(np.float32)
    n = len(o)
    return dict(ox=o[:, 0].copy(), oy=o[:, 1].copy(), oz=o[:, 2].copy(), dx=d[:, 0].copy(),
                dy=d[:, 1].copy(), dz=d[:, 2].copy(), tmin=np.zeros(n, np.float32),
                tmax=np.full(n, np.inf, np.float32))


def _aimed(p, ext, seed, axes=(0, 1, 2)):
    """Rays through the points p: along an axis, with zeros of both signs, and
    with one or both of the other components tiny (down to denormals)."""
    g = np.random.default_rng(seed)
    n = len(p)
    k = np.resize(axes, n)
    axis = np.zeros((n, 3))
    axis[np.arange(n), k] = np.where(np.arange(n) % 2, 1.0, -1.0)
    o = p - axis * ext * 0.75
    zero = np.where(np.arange(n) % 4 < 2, 0.0, -0.0)[:, None]
    tiny = 10.0 ** -g.uniform(4, 44, (n, 3)) * g.choice([-1.0, 1.0], (n, 3))
    mixed = np.where(g.random((n, 3)) < 0.5, tiny, zero)
    return concat_rays(_pack(o, np.where(axis == 0, zero, axis)),
                       _pack(o, np.where(axis == 0, tiny, axis)),
                       _pack(o, np.where(axis == 0, mixed, axis)))


def _check(ctx, O, geo, rays, hit_share):
    upload = ctx.upload_spheres if hasattr(geo, "cx") else ctx.upload_scene
    s = upload(geo)
    b = ctx.build_lbvh(s, _rq.MORTON_SCENE_AABB)
    saved = ctx.trace_config()
    try:
        ob = O.OracleBVH(geo, 1)
        o, oa = ob.closest(rays), ob.any(rays)
        assert (o["prim"] >= 0).mean() >= hit_share
        # the defaults, one whose stack entries carry distances, full refills
        for closest, any_, refill in ((saved[0], saved[1], 64), (12, 16, 16)):
            ctx.trace_config(closest, any_, refill)
            g = ctx.closest_hit(b, rays)
            bad = np.flatnonzero(g["prim"] != o["prim"])
            assert not len(bad), (closest, len(bad), bad[:5])
            for k in ("t", "u", "v"):
                assert np.array_equal(_bits(g[k]), _bits(o[k])), (closest, k)
            assert np.array_equal(ctx.any_hit(b, rays)["occ"], oa["occ"]), any_
        # few rays, walked by several lanes each
        few = {k: v[::41].copy() for k, v in rays.items()}
        assert np.array_equal(ctx.closest_hit(b, few)["prim"], o["prim"][::41])
        assert ctx.device_errors() == 0
    finally:
        ctx.trace_config(*saved)
        ctx.release(b)
        ctx.release(s)


def _soup(scale, offset=0.0):
    m = random_soup(700, 5, spread=2.0, size=0.2)
    x = (np.stack([m.vx, m.vy, m.vz]).astype(np.float64) * scale
         + np.array([[1.0], [-0.5], [0.25]]) * offset).astype(np.float32)
    return _rq.MeshArrays(x[0].copy(), x[1].copy(), x[2].copy(), m.idx)


def _points(mesh, n, seed):
    g = np.random.default_rng(seed)
    tri = np.stack([mesh.vx, mesh.vy, mesh.vz], 1).astype(np.float64)[mesh.idx.reshape(-1, 3)]
    w = g.dirichlet([1, 1, 1], n)
    w[: n // 4] = [1, 0, 0]
    return (tri[g.integers(0, len(tri), n)] * w[:, :, None]).sum(1)


# past 1e12 the triangle test itself overflows: no hits, but the same answers
@pytest.mark.parametrize("scale,offset", [
    (1e-4, 0), (1.0, 0), (1e6, 0), (1.5e7, 0), (3e7, 0), (1e8, 0), (1e9, 0), (3e10, 0), (1e11, 0),
    (1e12, 0), (1e15, 0), (1e18, 0), (1e25, 0), (10.0, 1e6), (1e7, 1e12), (1e8, 1e12)])
def test_axis_rays_at_every_scale(ctx, O, scale, offset):
    mesh = _soup(scale, offset)
    rays = _aimed(_points(mesh, 2000, 3), 4.0 * scale, 4)
    log(f"axis rays: scale {scale:g}, offset {offset:g}")
    _check(ctx, O, mesh, rays, 0.3 if 1.0 <= scale <= 1e12 else 0.0)


@pytest.mark.parametrize("ground", [1e4, 3e7, 1e8, 1e10, 1e13])
def test_axis_rays_over_a_ground_sphere(ctx, O, ground):
    """A small cloud above one huge sphere, the reference's kind of scene; the
    rays pass over it (what a ray down to it hits first is lost in the huge
    sphere's own rounding)."""
    g = np.random.default_rng(8)
    n = 500
    c = g.uniform(-3, 3, (n, 3)).astype(np.float32)
    r = g.uniform(0.05, 0.4, n).astype(np.float32)
    c = np.vstack([c, np.array([[0.0, -ground - 10.0, 0.0]], np.float32)])
    r = np.append(r, np.float32(ground))
    sph = _rq.SphereArrays(*(np.ascontiguousarray(c[:, k]) for k in range(3)), r,
                           np.zeros(3 * (n + 1), np.float32))
    at = g.integers(0, n, 2000)
    p = c[at].astype(np.float64) + g.normal(size=(2000, 3)) * r[at][:, None] * 0.4
    log(f"axis rays over a ground sphere of {ground:g}")
    _check(ctx, O, sph, _aimed(p, 8.0, 9, axes=(0, 2)), 0.5)


def test_axis_rays_in_a_batch(ctx, O):
    """The batch run's own walk."""
    meshes = [_soup(s) for s in (1.0, 3e7, 1e9)]
    items, keep, want = [], [], []
    try:
        for m, scale in zip(meshes, (1.0, 3e7, 1e9)):
            rays = _aimed(_points(m, 1500, 5), 4.0 * scale, 6)
            d = _rq.DeviceRays.from_host(ctx, rays)
            hits = {k: _rq.DeviceArray(ctx, 4 * d.n) for k in ("prim", "t")}
            occ = _rq.DeviceArray(ctx, d.n)
            items.append(dict(scene=ctx.upload_scene(m), rays=d, hits=hits, occ=occ))
            keep += [d, occ, *hits.values()]
            ob = O.OracleBVH(m, 1)
            want.append((ob.closest(rays), ob.any(rays)["occ"]))
        log("axis rays in a batch")
        batch = _rq.Batch(ctx, items)
        batch.run()
        ctx.sync()
        for it, (o, oa) in zip(items, want):
            n = it["rays"].n
            assert np.array_equal(it["hits"]["prim"].download(np.int32, n), o["prim"])
            assert np.array_equal(it["hits"]["t"].download(np.uint32, n), _bits(o["t"]))
            assert np.array_equal(it["occ"].download(np.uint8, n), oa)
        batch.close()
    finally:
        for k in keep:
            k.free()
        for it in items:
            ctx.release(it["scene"])
