"""GPU: several right-hand sides from host memory with outputs that lie over the inputs, shifted by whole columns:
every input counts as it was before the call.  Against the single-vector product (1e-12, as in the tests of the
16-wide launches)."""
import numpy as np
import pytest

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def system():
    P = np.random.default_rng(5).uniform(-1, 1, (2, 1500))
    g = h2w.Initialisation(2, 1500, 40, 1.0, 8, h2w.CHOICE_RBF, h2w.NESTED, points=P)
    g.tree_initialisation()
    return g


def _products(g, X):
    return np.stack([g.mat_vec_prod(np.ascontiguousarray(x)) for x in X])


def _columns(g, x, y, nrhs, ld):
    return h2w.lib().h2w_matvec_ex(g._h, h2w._ptr(x), h2w._ptr(y), nrhs, ld, h2w.FP64, h2w.ORDER_INPUT, h2w.HOST)


@pytest.mark.parametrize("shift", [0, 8, -8, 16])
def test_outputs_over_inputs(system, shift):
    g, N, nrhs = system, system.N, 40
    buf = np.random.default_rng(6).normal(size=(nrhs + abs(shift), N))
    x0, y0 = (0, shift) if shift >= 0 else (-shift, 0)
    want = _products(g, buf[x0:x0 + nrhs].copy())
    assert _columns(g, buf[x0:], buf[y0:], nrhs, N) == h2w.H2W_OK
    err = np.linalg.norm(buf[y0:y0 + nrhs] - want) / np.linalg.norm(want)
    assert err <= 1e-12

