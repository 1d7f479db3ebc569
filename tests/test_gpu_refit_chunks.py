"""The refit's boxes at the edges of its leaf chunks: every node's box equals
the oracle's bit for bit, and the wide records hold the exact boxes (checked by
their export), for sizes around one, two and many chunks and around the size
at which the chunks get larger; evenly spread leaves, all leaves under one code
(split by index) and trees as deep as the codes allow."""
import numpy as np
import pytest

from conftest import log
from helpers import duplicate_mesh, mesh_from, random_soup
from test_gpu_build import _check_build

pytestmark = pytest.mark.gpu


def _chain(n):
    """Triangles at distances 2^-k from a corner: a node a level."""
    k = np.arange(n) % 28
    p = 2.0 ** -k[:, None, None] * np.array([1, 1, 1]) + (np.arange(n) // 28)[:, None, None] * 1e-10
    v = p + np.array([[0, 0, 0], [1e-3, 0, 0], [0, 1e-3, 0]]) * 2.0 ** -k[:, None, None]
    return mesh_from(v.reshape(-1, 3), np.arange(3 * n))


MESHES = {"soup": lambda n: random_soup(n, n, spread=2.0, size=0.02), "one_code": duplicate_mesh,
          "chain": _chain}
SIZES = [1, 2, 64, 255, 256, 257, 258, 511, 512, 513, 769, 1025, 4001]


@pytest.mark.parametrize("kind", list(MESHES))
@pytest.mark.parametrize("n", SIZES)
def test_refit_chunk_edges(ctx, O, rq, kind, n):
    log(f"refit chunks {kind} n={n}")
    mesh = MESHES[kind](n)
    _check_build(ctx, O, rq, mesh, 1)
    if n > 1:
        s = ctx.upload_scene(mesh)
        b = ctx.build_lbvh(s, 1)
        try:
            assert ctx.export_wide(b, n)["links"].shape == (n - 1, 4)
        finally:
            ctx.release(b)
            ctx.release(s)


@pytest.mark.parametrize("n", [(1 << 19) - 1, 1 << 19, (1 << 19) + 257])
def test_refit_where_chunks_grow(ctx, O, rq, n):
    log(f"refit chunks n={n}")
    _check_build(ctx, O, rq, MESHES["soup"](n), 1)
