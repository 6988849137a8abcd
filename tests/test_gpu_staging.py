"""GPU: the staging that a handle keeps for host columns follows the columns of a call, not the 16 of a full pass."""
import numpy as np
import pytest
import torch

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def test_two_columns():
    N = 500000
    P = np.random.default_rng(5).uniform(-1, 1, (1, N))
    g = h2w.Initialisation(1, N, 256, 1.0, 6, h2w.CHOICE_IE, h2w.NESTED, points=P)
    g.tree_initialisation()
    X = np.random.default_rng(6).normal(size=(2, N))
    d = torch.from_numpy(X).cuda()
    y = torch.empty_like(d)
    # (the same product on device columns takes what the product itself needs)
    rc = h2w.lib().h2w_matvec_ex(g._h, d.data_ptr(), y.data_ptr(), 2, N, h2w.FP64, h2w.ORDER_INPUT, h2w.DEVICE)
    assert rc == h2w.H2W_OK
    free = torch.cuda.mem_get_info()[0]
    Y = g.matvec_multi(X)
    assert free - torch.cuda.mem_get_info()[0] <= 2 * X.nbytes + (4 << 20)
    assert np.linalg.norm(Y - y.cpu().numpy()) <= 1e-12 * np.linalg.norm(Y)
