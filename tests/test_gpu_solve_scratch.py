"""GPU: the device memory that a solve takes follows the steps it makes, not the limit on them."""
import numpy as np
import pytest
import torch

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def test_high_step_limit():
    N = 130000
    P = np.random.default_rng(5).uniform(-1, 1, (1, N))
    g = h2w.Initialisation(1, N, 64, 1.0, 8, h2w.CHOICE_IE, h2w.NESTED, points=P)
    g.tree_initialisation()
    b = g.mat_vec_prod(np.random.default_rng(6).uniform(-1, 1, N))
    x, st = g.gmres(b, None, 500, 1e-4, h2w.GMRES_FP64)
    free = torch.cuda.mem_get_info()[0]
    x, st = g.gmres(b, None, 1000000, 1e-4, h2w.GMRES_FP64)
    assert st["converged"]
    # (the Hessenberg columns' buffer holds two numbers per permitted step)
    assert free - torch.cuda.mem_get_info()[0] <= 64 << 20
