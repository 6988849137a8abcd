"""GPU: saving an operator while the calling thread captures a HIP graph on a stream of its own: the save uses only the
handle's stream, so that the capture stays valid, and the file is the one written outside of it."""
import numpy as np
import pytest
import torch

import h2weak_amd as h2w

pytestmark = pytest.mark.gpu


def test_save_under_capture(tmp_path):
    P = np.random.default_rng(5).uniform(-1, 1, (2, 1500))
    g = h2w.Initialisation(2, 1500, 40, 1.0, 8, h2w.CHOICE_RBF, h2w.NESTED, points=P)
    g.tree_initialisation()
    g.save(tmp_path / "outside")
    x = torch.ones(1000, device="cuda")
    y = torch.zeros(1000, device="cuda")
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        y.copy_(x * 3.0)
        g.save(tmp_path / "inside")
    for k in range(3):
        x.fill_(k + 1.0)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.all(y == 3.0 * (k + 1.0))
    assert (tmp_path / "inside").read_bytes() == (tmp_path / "outside").read_bytes()
