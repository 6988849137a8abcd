"""GPU: composite transfers that are not used take no place in a handle.  1D, uniform points at 1e-12: the transfers'
entries exceed the limit from the leaves up, so that the product's launches are those of the levels one by one.  Beside
the blocks that the product reads (padded to four rows and 256 bytes: less than a twentieth for ranks of 45 to 70)
the handle holds L and R of every skeleton and, per slot of the vector pool, its vectors, point and coordinates."""
import numpy as np
import pytest
import torch

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def test_refused_composites_take_no_memory():
    N = 250000
    P = np.random.default_rng(1).uniform(-1, 1, (1, N))
    torch.cuda.synchronize()
    g = h2w.Initialisation(1, N, 64, 1.0, 12, h2w.CHOICE_RBF, h2w.NESTED, points=P, fp32_shadow=0, ir_tol_pow=0)
    free = torch.cuda.mem_get_info()[0]
    g.tree_initialisation()
    held = free - torch.cuda.mem_get_info()[0]
    r = np.array([len(g.skeleton(1, j, b)[0]) for j in range(1, g.stats()["nlevels"] + 1) for b in range(2 ** j)], float)
    slots = 2 * N + 2 * r.sum()
    lists = 48 << 20  # work items and terms, those of the directed lists of the on-the-fly products among them
    most = 1.05 * g.stats()["stored_bytes_fp64"] + 16 * (r ** 2).sum() + slots * (8 + 4 + 4 + 3 * 16) + lists
    assert held <= most
