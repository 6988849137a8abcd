"""GPU: the factors in a saved file, formed from the pivots on the device eight at a time: L unit lower and R upper
triangular, and L R the kernel's values at the pivots.  Every entry of the elimination takes at most `rank` products and
subtractions, so |L R - K| <= 2 (rank + 2) eps |L| |R| entry for entry.  Ranks from one to well beyond a chunk of eight
and its multiples, files of one and of several copied chunks, families and pairs."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def _factors(path):
    """(Ir, Ic, L, R) of every skeleton of a file, and its points in input order."""
    d = path.read_bytes()
    at = 8
    dim, _, _, _, _, nL, _, _ = np.frombuffer(d, np.int32, 8, at)
    N = int(np.frombuffer(d, np.int64, 1, at + 32)[0])
    at += 48
    P = np.frombuffer(d, np.float64, dim * N, at).reshape(dim, N)
    at += 8 * dim * N
    out = []

    def take(dt, n):
        nonlocal at
        v = np.frombuffer(d[at:at + n * np.dtype(dt).itemsize], dt)
        at += v.nbytes
        return v

    def skeleton(r):
        Ir, Ic = take(np.int32, r), take(np.int32, r)
        L = take(np.float64, r * r).reshape(r, r).T
        R = take(np.float64, r * r).reshape(r, r).T
        if r:
            out.append((Ir, Ic, L, R))

    for _ in range(2 * (nL + 1)):
        for _ in range(int(take(np.int32, 1)[0])):
            skeleton(int(take(np.int32, 1)[0]))
            take(np.float64, int(take(np.int32, 1)[0]))
    for _ in range(int(take(np.int64, 1)[0])):
        skeleton(int(take(np.int32, 4)[3]))
    assert at == len(d) - 8
    return out, P


@pytest.mark.parametrize("case", [(1, 3000, 50, 10, h2w.SEMI_NESTED), (2, 3001, 40, 8, h2w.NESTED),
                                  (3, 9001, 40, 8, h2w.NESTED)], ids=lambda c: f"{c[0]}d-N{c[1]}-v{c[4]}")
def test_factors_of_a_file(case, tmp_path):
    dim, N, nmax, tp, var = case
    pts = np.random.default_rng(5).uniform(-1, 1, (dim, N))
    g = h2w.Initialisation(dim, N, nmax, 1.0, tp, h2w.CHOICE_IE, var, points=pts)
    g.tree_initialisation()
    g.save(tmp_path / "op")
    skels, P = _factors(tmp_path / "op")
    T = P[:, g.tree_order()]
    ranks = {len(s[0]) for s in skels}
    assert min(ranks) < 40 and max(ranks) > 16 and any(r % 8 for r in ranks)
    eps = np.finfo(float).eps
    for Ir, Ic, L, R in skels:
        r = len(Ir)
        assert np.array_equal(np.triu(L), np.eye(r)) and np.array_equal(np.tril(R, -1), np.zeros((r, r)))
        D = np.sqrt(((T[:, Ir, None] - T[:, None, Ic]) ** 2).sum(0))
        K = {1: np.log(D), 2: -np.log(D) / (2 * np.pi), 3: 1 / (4 * np.pi * D)}[dim]
        # (the kernel's own rounding: a few eps of an entry, of the logarithm's argument where that is near one)
        assert np.all(np.abs(L @ R - K) <= 2 * (r + 2) * eps * (np.abs(L) @ np.abs(R)) + 8 * eps * (1 + np.abs(K)))
