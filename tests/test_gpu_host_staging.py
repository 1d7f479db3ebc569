"""Host-array queries at the sizes where their staging changes: rays read and
results written in pinned memory by the kernel, copied whole, array by array,
and in more than one chunk. Every output equals the device query's, whichever
outputs are asked for, also right after a call of another size."""
import ctypes as C

import numpy as np
import pytest

import rq as _rq
from conftest import log
from helpers import RAY_FIELDS, concat_rays, random_rays, random_soup, rays_toward

pytestmark = pytest.mark.gpu


def _bits(a):
    return np.asarray(a, np.float32).view(np.uint32)


def _ptr(a):
    return a.ctypes.data_as(C.c_void_p) if a is not None else None


@pytest.mark.parametrize("n", [1, 65, 2047, 2048, 2049, (1 << 18) - 1, 1 << 18, (1 << 18) + 3,
                               (1 << 20) + 2049])
def test_host_query_staging(ctx, n):
    log(f"host query n={n}")
    half = (n + 1) // 2
    rays = concat_rays(rays_toward(half, 3), random_rays(n - half, 4))
    s = ctx.upload_scene(random_soup(3000, 5, spread=1.5, size=0.05))
    b = ctx.build_lbvh(s, 1)
    stream = ctx.stream_create()
    try:
        want, occ = ctx.closest_hit(b, rays), ctx.any_hit(b, rays)["occ"]
        few = {k: v[:7].copy() for k, v in rays.items()}
        for _ in range(2):
            g = ctx.closest_hit_host(b, rays)
            assert np.array_equal(g["prim"], want["prim"])
            for k in ("t", "u", "v"):
                assert np.array_equal(_bits(g[k]), _bits(want[k])), k
            assert np.array_equal(ctx.any_hit_host(b, rays), occ)
            m = min(n, 7)
            assert np.array_equal(ctx.closest_hit_host(b, few)["prim"], want["prim"][:m])
        # the primitive alone, and with gaps in the optional outputs
        r = _rq.Rays(*[_ptr(rays[k]) for k in RAY_FIELDS])
        for names in ((), ("v",), ("t", "v"), ("u",)):
            out = {k: np.full(n + 1, 7, np.int32 if k == "prim" else np.float32)
                   for k in ("prim", *names)}
            h = _rq.Hits(*[_ptr(out.get(k)) for k in ("prim", "t", "u", "v")])
            ctx._check(_rq.lib().rq_closest_hit_host(ctx.h, b, C.byref(r), n, C.byref(h), stream))
            assert np.array_equal(out["prim"][:n], want["prim"]) and out["prim"][n] == 7
            for k in names:
                assert np.array_equal(_bits(out[k][:n]), _bits(want[k])) and out[k][n] == 7, names
        assert ctx.device_errors() == 0
    finally:
        ctx.stream_destroy(stream)
        ctx.release(b)
        ctx.release(s)
