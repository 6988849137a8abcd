"""GPU: work lists at the edges of their rules: thousands of tiny items (one item per wave, counts that are no
multiple of four, empty boxes), leaves of one to a few points, and items split by columns.  The single-vector
product against dense FP64 rows (30 tol) and against the 16-wide product (other kernels, the same operator)."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu

# dim, N, n_max, tol_pow, choice, variant
CASES = [
    (1, 40001, 8, 10, h2w.CHOICE_RBF, h2w.NESTED),
    (1, 20003, 8, 10, h2w.CHOICE_IE, h2w.SEMI_NESTED),
    (2, 20011, 6, 8, h2w.CHOICE_IE, h2w.NESTED),
    (2, 9001, 40, 8, h2w.CHOICE_RBF, h2w.SEMI_NESTED),
    (3, 6007, 4, 6, h2w.CHOICE_RBF, h2w.NESTED),
    (3, 5003, 130, 8, h2w.CHOICE_IE, h2w.NON_NESTED),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}d-N{c[1]}-n{c[2]}-ch{c[4]}-v{c[5]}")
def test_products_agree(case):
    dim, N, nmax, tp, ch, var = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, var, points=P)
    g.tree_initialisation()
    X = np.random.default_rng(6).normal(size=(3, N))
    rows = np.sort(np.random.default_rng(7).choice(N, 600, replace=False))
    y = np.stack([g.mat_vec_prod(x) for x in X])
    d = g.dense_rows(rows, X[0])
    assert np.linalg.norm(y[0][rows] - d) <= 30 * 10.0 ** -tp * np.linalg.norm(d)
    scale = np.linalg.norm(y)
    assert np.linalg.norm(g.matvec_multi(X) - y) <= 1e-12 * scale
    # FP32: N-term sums of magnitude up to the row norms, rounded at 6e-8 each
    for prec in (h2w.FP32, h2w.FP32_OTF):
        z = np.stack([g.mat_vec_prod(x, precision=prec) for x in X])
        assert np.linalg.norm(z - y) <= 1e-5 * scale
