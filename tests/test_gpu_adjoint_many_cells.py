"""Fitting more small cells than the chip holds with two waves each (one wave a cell there): trace and
gradients are, bit for bit, those of the workgroup sizes asked for."""
import numpy as np
import pytest
import torch

from eden_amd import configs
from eden_amd.adjoint import Adjoint, trace

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,comps", [(2049, 3), (5000, 2)])
def test_many_small_cells(cells, comps):
    m = configs.random_trees(sizes=[comps] * cells, n_cells=cells, t_final_ms=0.5, seed=3, hh_everywhere=True)
    m.pulse_start = np.full(cells, 100.0, np.float32)
    res = []
    for threads in (0, 64, 128, 256):
        with Adjoint(m, threads_per_cell=threads) as adj:
            g0, a0 = adj.default_parameters()
            target = adj.forward(g0, a0).clone()
            g = (g0 * 1.1).clone().requires_grad_(True)
            a = a0.clone().requires_grad_(True)
            tr = trace(adj, g, a)
            ((tr - target) ** 2).mean().backward()
            res.append([x.detach().cpu().numpy() for x in (target, tr, g.grad, a.grad)])
    assert np.isfinite(res[0][2]).all() and np.abs(res[0][2]).max() > 0
    for r in res[1:]:
        for x, y in zip(r, res[0]):
            assert np.array_equal(x, y)
