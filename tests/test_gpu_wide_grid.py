"""The 4-wide nodes keep their boxes on a byte grid of their own: whatever the
scene's scale, position and flatness, the walk must still reach every triangle
that the exact boxes reach. Closest and any hits equal the oracle's bit for
bit, on rays that graze the boxes: along the axes (with zeros of both signs),
from points on box planes, and through vertices and edges. The export checks
each record's box against the exact one."""
import numpy as np
import pytest

from conftest import log
from helpers import concat_rays, random_soup

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _mesh(rq, kind):
    m = random_soup(700, 5, spread=2.0, size=0.2)
    x = np.stack([m.vx, m.vy, m.vz]).astype(np.float64)
    if kind == "unit":
        pass
    elif kind == "large":
        x *= 3e4
    elif kind == "far":  # coordinates a few hundred thousand times the triangles' size
        x = x * 8 + np.array([[3e5], [-2e5], [1e5]])
    elif kind == "flat":  # every triangle in one plane
        x[2] = -1.25
    elif kind == "slab":  # and in planes a rounding apart
        x[2] = -1.25 + 1e-6 * x[2]
    elif kind == "lattice":  # shared coordinates: many planes meet rays exactly
        x = np.round(x * 4) / 4
    elif kind == "two_scales":  # a huge triangle among small ones
        x[:, :3] = [[-9e4, 9e4, 0], [-9e4, -9e4, 9e4], [-7, -7, -7]]
    elif kind == "astronomic":  # coordinates past 2^100: no grid
        x[:, :3] = [[-3e31, 3e31, 0], [-3e31, -3e31, 3e31], [-7, -7, -7]]
    x = x.astype(np.float32)
    return rq.MeshArrays(x[0].copy(), x[1].copy(), x[2].copy(), m.idx)


def _rays(mesh, seed):
    g = np.random.default_rng(seed)
    v = np.stack([mesh.vx, mesh.vy, mesh.vz], 1).astype(np.float64)
    tri = v[mesh.idx.reshape(-1, 3)]
    n = 3000
    t = g.integers(0, len(tri), n)
    w = g.dirichlet([1, 1, 1], n)
    w[: n // 4] = [1, 0, 0]            # vertices
    w[n // 4: n // 2, 2] = 0           # edges
    w /= w.sum(1, keepdims=True)
    p = (tri[t] * w[:, :, None]).sum(1)
    ext = np.minimum(v.max(0) - v.min(0), 1e6)
    o = p + g.normal(size=(n, 3)) * ext * 0.7
    o[::5] = tri[g.integers(0, len(tri), len(o[::5])), 0]  # on a vertex: on box planes
    d = p - o
    k = np.arange(n) % 3
    axis = np.zeros((n, 3))
    axis[np.arange(n), k] = np.where(np.arange(n) % 2, 1.0, -1.0)
    oa = p - axis * ext[k][:, None] * 0.5
    zero = np.where(np.arange(n) % 4 < 2, 0.0, -0.0)[:, None]
    da = np.where(axis == 0, zero, axis)

    def pack(o, d, tmax):
        with np.errstate(all="ignore"):
            d = d / np.linalg.norm(d, axis=1, keepdims=True)
        o, d = o.astype(np.float32), d.astype(np.float32)
        return dict(ox=o[:, 0].copy(), oy=o[:, 1].copy(), oz=o[:, 2].copy(), dx=d[:, 0].copy(),
                    dy=d[:, 1].copy(), dz=d[:, 2].copy(), tmin=np.zeros(n, np.float32),
                    tmax=np.asarray(tmax, np.float32))
    far = np.full(n, np.inf)
    return concat_rays(pack(o, d, far), pack(oa, da, far),
                       pack(o, d, np.linalg.norm(d, axis=1) * 1.0001))


@pytest.mark.parametrize("kind", ["unit", "large", "far", "flat", "slab", "lattice", "two_scales",
                                  "astronomic"])
def test_grid_boxes_keep_every_hit(ctx, O, rq, kind):
    mesh = _mesh(rq, kind)
    rays = _rays(mesh, 11)
    log(f"wide grid {kind}: {mesh.ntri} triangles, {len(rays['ox'])} rays")
    s = ctx.upload_scene(mesh)
    b = ctx.build_lbvh(s, rq.MORTON_SCENE_AABB)
    try:
        if kind != "astronomic":
            w = ctx.export_wide(b, mesh.ntri)
            assert w["links"].shape == (mesh.ntri - 1, 4)
        ob = O.OracleBVH(mesh, 1)
        o, oa = ob.closest(rays), ob.any(rays)
        g = ctx.closest_hit(b, rays)
        assert np.array_equal(g["prim"], o["prim"])
        for k in ("t", "u", "v"):
            assert np.array_equal(_bits(g[k]), _bits(o[k])), k
        assert np.array_equal(ctx.any_hit(b, rays)["occ"], oa["occ"])
        if kind not in ("flat", "slab"):
            assert (o["prim"] >= 0).mean() > 0.3
        assert ctx.device_errors() == 0
    finally:
        ctx.release(b)
        ctx.release(s)
