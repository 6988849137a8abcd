"""GPU: the complex work lists at the edges of the complex GEMV: items of one row to more than a tile of 128, row
counts around the powers of two that set the lanes per column, thousands of tiny items (one per wave, no multiple of
four), one level.  Products against dense rows with entries on the fly, 30 tol."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu

# dim, N, n_max, tol_pow, choice, variant
CASES = [
    (2, 20011, 6, 8, h2w.CHOICE_HANKEL, h2w.NESTED),
    (2, 20011, 6, 6, h2w.CHOICE_HANKEL, h2w.SEMI_NESTED),
    (3, 6007, 4, 6, h2w.CHOICE_HELMHOLTZ, h2w.NESTED),
    (3, 5003, 130, 8, h2w.CHOICE_HELMHOLTZ, h2w.NON_NESTED),
    (3, 4001, 33, 6, h2w.CHOICE_HELMHOLTZ, h2w.SEMI_NESTED),
    (3, 257, 200, 8, h2w.CHOICE_HELMHOLTZ, h2w.NESTED),
    (2, 521, 520, 8, h2w.CHOICE_HANKEL, h2w.NESTED),
    (3, 1153, 1100, 8, h2w.CHOICE_HELMHOLTZ, h2w.SEMI_NESTED),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}d-N{c[1]}-n{c[2]}-v{c[5]}")
def test_products_against_dense_rows(case):
    dim, N, nmax, tp, ch, var = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, var, points=P)
    g.tree_initialisation()
    rng = np.random.default_rng(6)
    x = rng.normal(size=N) + 1j * rng.normal(size=N)
    rows = np.sort(rng.choice(N, min(N, 600), replace=False))
    y = g.mat_vec_prod(x)
    d = g.dense_rows(rows, x)
    assert np.linalg.norm(y[rows] - d) <= 30 * 10.0 ** -tp * np.linalg.norm(d)
