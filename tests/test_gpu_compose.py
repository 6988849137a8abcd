"""GPU: composite transfers (several levels near the root in one launch) only where they round as the chain does: the
linearity defect A(x + z) - A x - A z of products, relative to A x, for systems whose transfers have large entries
(1D, uniform points, tolerance 1e-12: 1e3 to 1e5) and small ones.  Chains measure up to 2e-13 for random x; composites
of such entries 1e-12."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("case", [(1, 70003, 64, 12, h2w.CHOICE_IE, 5e-13), (1, 100000, 64, 12, h2w.CHOICE_RBF, 6e-14),
                                  (1, 2048, 64, 12, h2w.CHOICE_RBF, 5e-15), (2, 10000, 30, 12, h2w.CHOICE_IE, 5e-15)],
                         ids=lambda c: f"{c[0]}d-N{c[1]}")
def test_linearity(case):
    dim, N, nmax, tp, ch, tol = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, h2w.NESTED, points=P)
    g.tree_initialisation()
    rng = np.random.default_rng(6)
    x, z = rng.normal(size=N), 1e-2 * rng.normal(size=N)
    ax = g.mat_vec_prod(x)
    assert np.linalg.norm(g.mat_vec_prod(x + z) - ax - g.mat_vec_prod(z)) <= tol * np.linalg.norm(ax)
