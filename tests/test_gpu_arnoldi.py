"""GPU: the fused Arnoldi passes at the edges of their rules: rows that are no multiple of a workgroup's, the row
counts where its rows per thread change, columns in groups of eight, beyond the 16384 sums that the last workgroup
takes itself and beyond one chunk of 128.  The oracle is GMRES on the host (modified Gram-Schmidt twice, Givens
rotations) over the same products.  The residual that the recurrence reports is a product of the rotations' sines,
each known to rounding times ||A|| / h(j+1, j) (at most 1e-12 here), so that both agree to 1e-6 of themselves also
where the steps go on far below the products' rounding."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu

# dim, N, n_max, tol_pow, choice, steps
CASES = [
    (3, 255, 40, 8, h2w.CHOICE_IE, 7),
    (3, 513, 40, 8, h2w.CHOICE_IE, 9),
    (1, 131071, 64, 10, h2w.CHOICE_RBF, 8),
    (1, 131073, 64, 10, h2w.CHOICE_RBF, 70),
    (1, 262145, 64, 10, h2w.CHOICE_RBF, 17),
    (1, 524801, 64, 10, h2w.CHOICE_RBF, 66),
    (2, 1500, 40, 8, h2w.CHOICE_RBF, 530),
]


def host_residual(mv, b, steps):
    V = np.zeros((steps + 1, b.size))
    V[0] = b / np.linalg.norm(b)
    rot, res = [], 1.0
    for j in range(steps):
        w = mv(V[j])
        h = np.zeros(j + 1)
        for _ in range(2):
            for i in range(j + 1):
                c = V[i] @ w
                h[i] += c
                w -= c * V[i]
        nw = np.linalg.norm(w)
        V[j + 1] = w / nw
        for i, (c, s) in enumerate(rot):
            h[i], h[i + 1] = c * h[i] + s * h[i + 1], -s * h[i] + c * h[i + 1]
        r = np.hypot(h[j], nw)
        rot.append((h[j] / r, nw / r))
        res *= nw / r
    return res


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}d-N{c[1]}-k{c[5]}")
def test_same_steps_as_on_the_host(case):
    dim, N, nmax, tp, ch, steps = case
    P = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, ch, h2w.NESTED, points=P)
    g.tree_initialisation()
    b = np.random.default_rng(6).normal(size=N)
    x, st = g.gmres(b, np.zeros(N), steps, 1e-300, h2w.GMRES_FP64)
    # (the last case ends early, when the reported residual passes 1e-300)
    assert st["iterations"] == steps or st["converged"]
    assert np.linalg.norm(b - g.mat_vec_prod(x)) <= max(2 * st["resid"], 1e-10) * np.linalg.norm(b)
    res = host_residual(g.mat_vec_prod, b, st["iterations"])
    assert abs(st["resid"] - res) <= 1e-6 * res
