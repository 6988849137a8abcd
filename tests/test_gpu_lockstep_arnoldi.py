"""GPU: the lockstep Arnoldi passes at the edges of their rules: slots that are no multiple of a block's, blocks of
several hundred slots, more columns than a pass keeps in registers (24), systems of different sizes whose columns stop
at different steps.  The same solves one by one (other kernels): 16 columns against h2w_gmres, to 10 times the
residual tolerance in the solution (well conditioned systems, checked by the residuals), with the same iteration
counts up to one (a residual within rounding of the tolerance)."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def _system(dim, N, nmax, tp, ch, seed):
    P = np.random.default_rng(seed).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, h2w.NESTED, points=P)
    g.tree_initialisation()
    return g


def _check(g, B, X, st, tol):
    for b, x, s in zip(B, X, st):
        assert s["converged"]
        assert np.linalg.norm(b - g.mat_vec_prod(x)) <= 2 * tol * np.linalg.norm(b)
        y, sy = g.gmres(b, None, 300, tol, h2w.GMRES_FP64)
        assert abs(s["iterations"] - sy["iterations"]) <= 1
        assert np.linalg.norm(x - y) <= 10 * tol * np.linalg.norm(y)


@pytest.mark.parametrize("case", [(3, 1031, 40, 10, h2w.CHOICE_IE, 1e-9), (2, 3001, 40, 10, h2w.CHOICE_IE, 1e-10),
                                  (2, 70001, 64, 8, h2w.CHOICE_IE, 1e-8)], ids=lambda c: f"{c[0]}d-N{c[1]}")
def test_one_system(case):
    g = _system(*case[:5], 5)
    B = np.random.default_rng(6).normal(size=(16, g.N))
    B[3] = g.mat_vec_prod(np.ones(g.N))  # (from the starting guess itself: converged at once)
    X, st = g.gmres_multi(B, None, 300, case[5], h2w.GMRES_FP64)
    _check(g, B, X, st, case[5])


def test_batch_of_unequal_systems():
    G = [_system(3, 700, 40, 10, h2w.CHOICE_IE, 7), _system(2, 5003, 64, 10, h2w.CHOICE_IE, 8),
         _system(3, 9001, 64, 10, h2w.CHOICE_RBF, 9)]
    B = [np.random.default_rng(10 + k).normal(size=(3, g.N)) for k, g in enumerate(G)]
    X, st = h2w.Batch(G).gmres(B, None, 300, 1e-9, h2w.GMRES_FP64)
    for g, b, x, s in zip(G, B, X, st):
        _check(g, b, x, s, 1e-9)
