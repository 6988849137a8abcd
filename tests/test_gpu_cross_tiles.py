"""GPU: the batched cross at the edges of its 512-entry tiles.  Jittered 1D points put exactly N / 2 points
in each box of level 1, whose vertex block is then N / 2 x N / 2: one entry short of a tile, a whole tile,
one entry into the next, and the same at two tiles.  Skeletons are the oracle's box for box, on the first
assembly and on a second one of the same handle (which reuses nothing of the first)."""
import numpy as np
import pytest

import h2weak_amd as h2w
import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("half", [511, 512, 513, 1023, 1025])
@pytest.mark.parametrize("variant", [h2w.NESTED, h2w.SEMI_NESTED])
def test_blocks_at_tile_edges(half, variant):
    N = 2 * half
    x = (-1.0 + (2.0 * np.arange(N) + 1.0) / N + np.random.default_rng(half).uniform(-0.4, 0.4, N) / N)[None, :]
    o = oracle.Oracle(1, N, 32, 1.0, 10, 1, variant, points=x)
    o.tree_initialisation()
    g = h2w.Initialisation(1, N, 32, 1.0, 10, h2w.CHOICE_RBF, variant, points=x)
    xt = np.random.default_rng(1).normal(size=N)
    yo = o.mat_vec_prod(xt)
    for _ in range(2):
        g.tree_initialisation()
        if variant == h2w.NESTED:
            for j in range(1, o.nlevels + 1):
                for b in range(2 ** j):
                    assert g.skeleton(1, j, b) == o.pivots(1, j, b), (j, b)
        assert g.stats()["memory"] == o.memory
        assert np.linalg.norm(g.mat_vec_prod(xt) - yo) <= 1e-12 * np.linalg.norm(yo)
