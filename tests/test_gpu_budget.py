"""What creation takes of a context's HBM budget: a program sized to a budget keeps
working when kernels are compiled for more waves, whose stack overflow areas are
larger. The sums are those of 32-bit entries (64-bit where an entry carries its
distance) over the grids the kernels can have on 256 compute units."""
import numpy as np
import pytest

import rq as _rq
from conftest import log

pytestmark = pytest.mark.gpu

MB = 1 << 20


def test_context_in_240_mb():
    log("context in 240 MB")
    _rq.Context(0, 240 * MB).close()


def test_context_with_two_more_streams_in_721_mb():
    """A stream's first traversal allocates an overflow area of its own."""
    log("streams in 721 MB")
    c = _rq.Context(0, 721 * MB)
    try:
        s = c.upload_scene(_rq.soup(1000, 1))
        b = c.build_lbvh(s, _rq.MORTON_SCENE_AABB)
        rays = {k: np.zeros(64, np.float32) for k in _rq.RAY_FIELDS}
        d, prim = _rq.DeviceRays.from_host(c, rays), _rq.DeviceArray(c, 256)
        for _ in range(2):
            c.closest_hit_dev(b, d, {"prim": prim}, stream=c.stream_create())
        c.sync()
        assert c.device_errors() == 0
    finally:
        c.close()


def test_batch_in_493_mb():
    log("batch in 493 MB")
    c = _rq.Context(0, 493 * MB)
    try:
        s = c.upload_scene(_rq.soup(1000, 1))
        rays = {k: np.zeros(1000, np.float32) for k in _rq.RAY_FIELDS}
        d, prim = _rq.DeviceRays.from_host(c, rays), _rq.DeviceArray(c, 4000)
        _rq.Batch(c, [dict(scene=s, rays=d, hits={"prim": prim}, occ=None)]).close()
    finally:
        c.close()


def test_server_in_505_mb():
    log("server in 505 MB")
    _rq.Server(0, mesh_slots=2, slot_tris=10000, arena_bytes=1 << 24, hbm_budget=505 * MB).close()


@pytest.mark.parametrize("mode", [_rq.RENDER_SHADE, _rq.RENDER_OCCLUSION])
def test_renderer_takes_what_it_needs_only(O, mode):
    """A renderer, and then an allocation that just fits beside what it needs."""
    p = _rq.render_defaults()
    p.width, p.height, p.camera, p.mode = 1920, 1080, _rq.CAMERA_PHILOX, mode

    def enough(budget):
        c = _rq.Context(0, budget)
        try:
            _rq.Renderer(c, p).close()
            return True
        except _rq.RQError:
            return False
        finally:
            c.close()
    lo, hi = 252 * MB, 1024 * MB
    while hi - lo > 4096:
        mid = (lo + hi) // 2
        lo, hi = (lo, mid) if enough(mid) else (mid, hi)
    mesh = _rq.icosphere(3, 2, center=(0, 0, -5))
    room = 8 * MB
    log(f"renderer mode {mode} in {hi} bytes")
    c = _rq.Context(0, hi + room)
    try:
        ren = _rq.Renderer(c, p)
        a = _rq.DeviceArray(c, room)
        a.free()
        s = c.upload_scene(mesh)
        b = c.build_lbvh(s, _rq.MORTON_SCENE_AABB)
        first = None
        for _ in range(2):  # a read leaves nothing behind that the next frame uses
            ren.frame(b)
            rgb, ppm = ren.image()
            g = ren.samples()
            assert np.array_equal(ppm, O.resolve_ppm(g["rgb"], 1920 * 1080, 1))
            first = first if first is not None else (rgb, g)
            assert np.array_equal(rgb, first[0]) and np.array_equal(g["hit0"], first[1]["hit0"])
        assert np.array_equal(ren.image()[1], ppm)
        ren.close()
    finally:
        c.close()
