"""Batch runs at the edges of the build phases' tiles and of the trace queue:
mesh sizes around a wave, a sort tile, a refit chunk and a Morton / Karras
tile, batches whose phases have no items, and queues with fewer items than
segments, than waves, and far more. Trees and answers equal the per-mesh
path's bit for bit, over eager runs and graph replays in turn."""
import pytest

import rq as _rq
from conftest import log
from helpers import random_soup
from test_gpu_batch import Setup

pytestmark = pytest.mark.gpu


def _case(n, rays, closest=True, anyq=True):
    return (f"soup{n}", lambda: random_soup(n, n, spread=1.5, size=0.05), rays, closest, anyq)


BATCHES = {
    "one_tri_one_ray": [_case(1, (1, 0), True, False)],
    "one_item": [_case(300, (200, 0), False, True)],
    "no_spanning_nodes": [_case(n, (64, 64)) for n in (1, 2, 63, 65, 255)],
    "tile_edges": [_case(n, (300, 300)) for n in (256, 257, 1023, 1024, 1025, 2047, 2049, 4095,
                                                  4096, 4097, 8193)],
    "one_mesh_many_items": [_case(5000, (40000, 40000))],
    "no_rays": [_case(1500, (0, 0)), _case(2, (0, 0))],
}


@pytest.mark.parametrize("mode", [_rq.MORTON_SCENE_AABB, _rq.MORTON_REF_AFFINE])
@pytest.mark.parametrize("name", list(BATCHES))
def test_batch_edges(ctx, name, mode):
    log(f"batch {name} mode {mode}")
    st = Setup(ctx, mode, BATCHES[name])
    try:
        for rep in range(4):
            st.clear()
            (st.batch.run_graph if rep % 2 else st.batch.run)()
            st.check(st.results(), f"run {rep}")
            assert st.batch.errors() == 0
            ph = st.batch.phase_ms()
            assert all(v >= 0.0 for v in ph.values()), ph
        for waves in (8, 4):
            st.batch.build_waves(waves)
            st.clear()
            st.batch.run()
            st.check(st.results(), f"{waves} waves")
        st.check_trees()
        assert ctx.device_errors() == 0
    finally:
        st.close()
