"""GPU: the 16-wide fused launch at the edges of its rules: row counts around a slab (16, 32, 64 rows in FP64, up to 128
in FP32), leaves of more than one row tile, items of more than 64 terms, groups past a term's end, one to 17
right-hand sides.  Against the single-vector product (other kernels, the same stored operator): sums of N terms of
the same products in another order, 1e-12 in FP64 and 1e-5 in FP32 relative to the product."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu

# dim, N, n_max, tol_pow, choice, variant, right-hand sides
CASES = [
    (3, 9001, 4, 4, h2w.CHOICE_RBF, h2w.NESTED, 3),
    (3, 4096, 8, 6, h2w.CHOICE_IE, h2w.NON_NESTED, 16),
    (2, 9001, 17, 6, h2w.CHOICE_RBF, h2w.NESTED, 16),
    (2, 9001, 33, 8, h2w.CHOICE_IE, h2w.SEMI_NESTED, 5),
    (3, 5003, 65, 8, h2w.CHOICE_IE, h2w.NESTED, 17),
    (3, 5003, 140, 8, h2w.CHOICE_RBF, h2w.NESTED, 16),
    (2, 9001, 600, 10, h2w.CHOICE_RBF, h2w.NON_NESTED, 2),
    (1, 30011, 130, 10, h2w.CHOICE_RBF, h2w.NESTED, 16),
]


def _system(case):
    dim, N, nmax, tp, ch, var, _ = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, var, points=P)
    g.tree_initialisation()
    return g


def _agree(Z, g, X, prec, tol):
    y = np.stack([g.mat_vec_prod(x, precision=prec) for x in X])
    assert np.linalg.norm(Z - y) <= tol * np.linalg.norm(y)


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}d-N{c[1]}-n{c[2]}-v{c[5]}-r{c[6]}")
def test_products_agree(case):
    g = _system(case)
    X = np.random.default_rng(6).normal(size=(case[6], case[1]))
    for prec, tol in ((h2w.FP64, 1e-12), (h2w.FP32, 1e-5), (h2w.FP32_INNER, 1e-5)):
        if prec == h2w.FP32_INNER and case[3] <= 6:  # (no inner operator at its own tolerance of 1e-6)
            continue
        _agree(g.matvec_multi(X, precision=prec), g, X, prec, tol)


def test_batch_agrees():
    cs = [CASES[2], CASES[4], CASES[7]]
    G = [_system(c) for c in cs]
    X = [np.random.default_rng(6).normal(size=(5, c[1])) for c in cs]
    Y = h2w.Batch(G).matvec(X)
    for g, x, y in zip(G, X, Y):
        _agree(y, g, x, h2w.FP64, 1e-12)


def test_host_columns_with_gaps():
    g = _system(CASES[4])
    N, nrhs, ld = g.N, 19, g.N + 7
    X = np.full((nrhs, ld), np.nan)
    X[:, :N] = np.random.default_rng(6).normal(size=(nrhs, N))
    Y = np.full((nrhs, ld), -1.0)
    rc = h2w.lib().h2w_matvec_ex(g._h, h2w._ptr(X), h2w._ptr(Y), nrhs, ld, h2w.FP64, h2w.ORDER_INPUT, h2w.HOST)
    assert rc == h2w.H2W_OK
    _agree(Y[:, :N], g, np.ascontiguousarray(X[:, :N]), h2w.FP64, 1e-12)
    assert np.all(Y[:, N:] == -1.0)
