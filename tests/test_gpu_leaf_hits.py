"""Hits that the primitive test accepts by its rounding although the ray misses
the primitive's box. A wide node's box on the grid is larger than the exact
one, so the wide walk itself has to answer for the ray that hits the exact box;
a tree of one primitive has no box to miss. Answers equal the binary walk's and
the oracle's bit for bit."""
import numpy as np
import pytest

import rq as _rq
from conftest import log
from helpers import mesh_from

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _pack(o, d, tmax=None):
    o, d = np.asarray(o).astype(np.float32), np.asarray(d).astype(np.float32)
    n = len(o)
    return dict(ox=o[:, 0].copy(), oy=o[:, 1].copy(), oz=o[:, 2].copy(), dx=d[:, 0].copy(),
                dy=d[:, 1].copy(), dz=d[:, 2].copy(), tmin=np.zeros(n, np.float32),
                tmax=np.full(n, np.inf, np.float32) if tmax is None else
                np.asarray(tmax, np.float32))


def _check(ctx, b, rays, o, oa):
    saved = ctx.trace_config()
    try:
        for closest, any_, refill in ((saved[0], saved[1], 64), (0, 0, 64), (12, 16, 16)):
            ctx.trace_config(closest, any_, refill)
            g = ctx.closest_hit(b, rays)
            bad = np.flatnonzero(g["prim"] != o["prim"])
            assert not len(bad), (closest, len(bad), bad[:5])
            for k in ("t", "u", "v"):
                assert np.array_equal(_bits(g[k]), _bits(o[k])), (closest, k)
            bad = np.flatnonzero(ctx.any_hit(b, rays)["occ"] != oa["occ"])
            assert not len(bad), (any_, len(bad), bad[:5])
        assert ctx.device_errors() == 0
    finally:
        ctx.trace_config(*saved)


@pytest.mark.parametrize("n", [1, 2])
@pytest.mark.parametrize("distance", [3.0, 40.0, 400.0])
def test_grazing_a_distant_sphere(ctx, O, n, distance):
    """Rays around the outline of one sphere (no box), and of one of two."""
    g = np.random.default_rng(int(distance) + n)
    m, r = 60000, 0.05
    c = np.float32([[0.0, 0.0, -distance], [5.0, 0.0, -distance]])[:n]
    sph = _rq.SphereArrays(*(np.ascontiguousarray(c[:, k]) for k in range(3)),
                           np.full(n, r, np.float32), np.zeros(3 * n, np.float32))
    a = g.uniform(0, 2 * np.pi, m)
    at = r * g.uniform(0.9, 1.6, m)
    p = c[0] + np.stack([at * np.cos(a), at * np.sin(a), np.zeros(m)], 1)
    p[::3, :2] = c[0][:2] + g.uniform(-1.5 * r, 1.5 * r, (len(p[::3]), 2))
    o = np.zeros((m, 3))
    o[::2] = p[::2] + np.float32([0.0, 0.0, distance])  # parallel ones
    rays = _pack(o, (p - o) / np.linalg.norm(p - o, axis=1, keepdims=True))
    log(f"grazing {n} spheres at {distance:g}")
    s = ctx.upload_spheres(sph)
    b = ctx.build_lbvh(s, _rq.MORTON_SCENE_AABB)
    try:
        ob = O.OracleBVH(sph, 1)
        want = ob.closest(rays)
        assert 0.1 < (want["prim"] >= 0).mean() < 0.99
        if n == 1 and distance > 3:  # hits that a box would take away
            f = O.closest_brute(sph, rays, box_filter=True)
            assert ((f["prim"] < 0) & (want["prim"] >= 0)).any()
        _check(ctx, b, rays, want, ob.any(rays))
    finally:
        ctx.release(b)
        ctx.release(s)


def _triangles(g, n, aspect, offset):
    c = g.uniform(-12, 12, (n, 3)) + offset
    a = g.normal(size=(n, 3))
    a /= np.linalg.norm(a, axis=1, keepdims=True)
    e = g.normal(size=(n, 3))
    e -= (e * a).sum(1, keepdims=True) * a
    e /= np.linalg.norm(e, axis=1, keepdims=True)
    v = np.stack([c, c + a, c + a * g.uniform(0, 1, (n, 1)) + e * aspect], 1)
    flat = np.arange(n) % 2 == 0  # half of them in a plane of two axes
    k = np.arange(n) % 3
    for q in (1, 2):
        v[flat, q, k[flat]] = v[flat, 0, k[flat]]
    return v.astype(np.float32)


@pytest.mark.parametrize("length", [1e-3, 1.0, 1e3, "segment"])
@pytest.mark.parametrize("distance,aspect,offset", [
    (2.0, 1.0, 0.0), (30.0, 0.1, 100.0), (100.0, 1.0, 0.0), (3000.0, 1.0, 10.0), (3000.0, 1e-2, 0.0),
    (1e5, 1.0, 0.0), (1e6, 1.0, 1e3)])
def test_triangle_hits_outside_the_box(ctx, O, length, distance, aspect, offset):
    """Rays at vertices and edges, nearly or exactly parallel to axis planes (where
    a box forgives least), with directions of other lengths than one; segment:
    to the point aimed at, where t is 1 whatever the distance."""
    g = np.random.default_rng(int(distance) + int(offset))
    n = 60000
    v = _triangles(g, 64, aspect, offset)
    w = g.dirichlet([1, 1, 1], n)
    w[: n // 2] = [1, 0, 0]
    w[n // 2: 5 * n // 6, 2] = 0
    w /= w.sum(1, keepdims=True)
    t = g.integers(0, len(v), n)
    p = (v[t].astype(np.float64) * w[:, :, None]).sum(1)
    # across the triangle, or nearly along it
    nrm = np.cross((v[:, 1] - v[:, 0]).astype(np.float64), v[:, 2] - v[:, 0])[t]
    nrm /= np.linalg.norm(nrm, axis=1, keepdims=True)
    d = g.normal(size=(n, 3))
    along = np.where(g.random(n) < 0.5, 1 - 10.0 ** -g.uniform(0, 3, n), 0.0)[:, None]
    d -= (d * nrm).sum(1, keepdims=True) * nrm * along
    k = g.integers(0, 3, n)
    d[np.arange(n), k] *= np.where(g.random(n) < 0.3, 0.0, 10.0 ** -g.uniform(1, 9, n))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    o = (p - d * distance).astype(np.float32)
    step = g.integers(-3, 4, (n, 3)) * (np.abs(o) > 1e-20)  # a few roundings aside
    o = (o.view(np.int32) + step.astype(np.int32)).view(np.float32)
    if length == "segment":
        rays = _pack(o, d * distance, np.where(np.arange(n) % 3, 1.5, 1.00002))
    else:
        rays = _pack(o, d * length)
    mesh = mesh_from(v, np.arange(3 * len(v)))
    log(f"triangle hits outside the box: |d| {length}, distance {distance:g}, aspect {aspect:g}, "
        f"offset {offset:g}")
    s = ctx.upload_scene(mesh)
    b = ctx.build_lbvh(s, _rq.MORTON_SCENE_AABB)
    try:
        ob = O.OracleBVH(mesh, 1)
        want = ob.closest(rays)
        assert (want["prim"] >= 0).mean() > 0.05
        # the inputs do hold hits that only the test's rounding makes
        assert (O.closest_brute(mesh, rays)["prim"] != want["prim"]).sum() >= 3
        _check(ctx, b, rays, want, ob.any(rays))
    finally:
        ctx.release(b)
        ctx.release(s)
