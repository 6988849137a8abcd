"""GPU: composite transfers across a box without a skeleton.  Clustered points give a box whose far partners are all
empty (no skeleton) between descendants, a parent and a grandparent that have one: the block of a descendant and the
parent is never formed, and the grandparent's is formed from it.  Freed device memory is filled with NaN before the
assembly, so that anything read before it is written shows.  Against the oracle's product over the same skeletons
(its parity bound, the tolerance of the crosses)."""
import ctypes

import numpy as np
import pytest

import h2weak_amd as h2w
import oracle

pytestmark = pytest.mark.gpu


def _clusters():
    """Points by (level, column, row, number of points) of the boxes that hold them, in [-1, 1]^2."""
    rng = np.random.default_rng(1)
    out = []
    for j, ix, iy, n in [(4, 4, 8, 120), (4, 5, 8, 60), (4, 3, 8, 60), (2, 3, 2, 200), (2, 3, 3, 200), (3, 5, 4, 80)]:
        w = 2.0 / 2 ** j
        out.append(np.array([[-1 + ix * w], [-1 + iy * w]]) + w * rng.uniform(0.02, 0.98, (2, n)))
    return np.concatenate(out, 1)


def _fill_free_memory():
    hip = ctypes.CDLL("libamdhip64.so.7")
    hip.hipMalloc.argtypes = [ctypes.c_void_p, ctypes.c_size_t]
    hip.hipMemset.argtypes = [ctypes.c_void_p, ctypes.c_int, ctypes.c_size_t]
    hip.hipFree.argtypes = [ctypes.c_void_p]
    held = []
    for size in [1 << k for k in range(12, 22)] * 16:
        p = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(p), size) == 0
        assert hip.hipMemset(p, 0xFF, size) == 0
        held.append(p)
    assert hip.hipDeviceSynchronize() == 0
    for p in held:
        assert hip.hipFree(p) == 0


@pytest.mark.parametrize("choice", [h2w.CHOICE_IE, h2w.CHOICE_RBF])
def test_box_without_a_skeleton(choice):
    P = _clusters()
    N = P.shape[1]
    o = oracle.Oracle(2, N, 8, 1.0, 8, choice, h2w.NESTED, points=P, nlevels=5)
    o.tree_initialisation()
    ranks = [[len(o.pivots(0, j, b)[0]) for b in range(4 ** j)] for j in range(6)]
    gaps = [b for b in range(4 ** 4) if ranks[4][b] == 0 and any(ranks[5][4 * b:4 * b + 4]) and ranks[3][b // 4]
            and ranks[2][b // 16]]
    assert gaps  # (the points make what the test is about)
    _fill_free_memory()
    g = h2w.Initialisation(2, N, 8, 1.0, 8, choice, h2w.NESTED, points=P, nlevels=5)
    g.tree_initialisation()
    x = np.random.default_rng(2).normal(size=N)
    y, yo = g.mat_vec_prod(x), o.mat_vec_prod(x)
    err = np.linalg.norm(y - yo) / np.linalg.norm(yo)
    assert err <= 1e-8
