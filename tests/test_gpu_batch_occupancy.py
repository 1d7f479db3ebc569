"""rq_batch_occupancy: what it reports is counted by the run itself."""
import pytest

import rq as _rq
from conftest import log
from helpers import random_rays

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rays", [64, 5000])
def test_occupancy_counts_the_runs_own_blocks(ctx, rays):
    """The trace blocks of a run are counted on the device: none before it, then the
    launch's whole grid, which a batch of few items keeps small."""
    log(f"batch occupancy, {rays} rays")
    s = ctx.upload_scene(_rq.icosphere(3, 2))
    d = _rq.DeviceRays.from_host(ctx, random_rays(rays, 3))
    prim = _rq.DeviceArray(ctx, 4 * rays)
    batch = _rq.Batch(ctx, [dict(scene=s, rays=d, hits={"prim": prim}, occ=None)])
    try:
        tile = batch.config()[1]
        items = (rays + tile - 1) // tile
        want = 8 * ((items + 31) // 32)  # a wave for each item, on every XCD
        assert batch.occupancy() == (0, want)
        for run in (batch.run, batch.run_graph, batch.run_graph, batch.run):
            run()
            assert batch.occupancy() == (want, want)
    finally:
        batch.close()
        d.free()
        prim.free()
        ctx.release(s)
