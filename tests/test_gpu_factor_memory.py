"""GPU: the skeletons' factors L and R take no device memory beside an assembled operator (they are formed from the
pivots where an inner operator or a saved file needs them), and what is formed is what the cross approximation
produced: an inner operator rebuilt at its own tolerance equals the one of the assembly, which took the cross's factors
(products to the rounding of FP32 sums in another order, 1e-6, as in the tests of saved operators)."""
import numpy as np
import pytest
import torch

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def test_device_memory():
    N = 250000
    P = np.random.default_rng(1).uniform(-1, 1, (1, N))
    g = h2w.Initialisation(1, N, 64, 1.0, 12, h2w.CHOICE_RBF, h2w.NESTED, points=P, fp32_shadow=0, ir_tol_pow=0)
    free = torch.cuda.mem_get_info()[0]
    g.tree_initialisation()
    held = free - torch.cuda.mem_get_info()[0]
    r = np.array([len(g.skeleton(1, j, b)[0]) for j in range(1, g.stats()["nlevels"] + 1) for b in range(2 ** j)], float)
    slots = 2 * N + 2 * r.sum()
    lists = 48 << 20  # work items and terms, those of the directed lists of the on-the-fly products among them
    # (blocks padded to four rows and 256 bytes; per slot its vectors, point and coordinates)
    assert held <= 1.05 * g.stats()["stored_bytes_fp64"] + slots * (8 + 4 + 4 + 3 * 16) + lists


@pytest.mark.parametrize("case", [(1, 4096, 64, 12, h2w.CHOICE_RBF), (2, 5003, 40, 10, h2w.CHOICE_IE),
                                  (3, 9001, 64, 8, h2w.CHOICE_RBF)], ids=lambda c: f"{c[0]}d-N{c[1]}")
def test_inner_operator_again(case):
    dim, N, nmax, tp, ch = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, h2w.NESTED, points=P)
    g.tree_initialisation()
    x = np.random.default_rng(6).normal(size=N)
    y = g.mat_vec_prod(x, precision=h2w.FP32_INNER)
    g.set_inner_tolerance(5.0)
    g.set_inner_tolerance(6.0)
    z = g.mat_vec_prod(x, precision=h2w.FP32_INNER)
    assert np.abs(z - y).max() <= 1e-6 * np.abs(y).max()
