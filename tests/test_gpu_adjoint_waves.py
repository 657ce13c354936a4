"""The adjoint kernels with a wave that solves beside waves that advance gates: the trace matches
the oracle's double-precision flavour, and trace and gradients are the same bit for bit with one
wave, two and four, with stored and recomputed step records: cells of 2 compartments, chains of
more rounds than headers are held, wide nodes, and more gates than a lane keeps derivatives for."""
import numpy as np
import pytest
import torch

from eden_amd import configs
from eden_amd.adjoint import Adjoint, trace
from oracle import oracle

pytestmark = pytest.mark.gpu


def _parents(shape):
    if shape == "small":
        return [np.array([-1, 0], np.int32), np.array([-1, 0, 0, 1, 1, 2], np.int32)]
    if shape == "chain":
        return [np.arange(-1, n - 1, dtype=np.int32) for n in (63, 64, 66, 70, 90)]
    if shape == "wide":
        return [np.array([-1] + [i // 6 for i in range(79)], np.int32), np.array([-1] + [0] * 69, np.int32)]
    return [np.array([-1] + [i // 2 for i in range(129)], np.int32), np.array([-1] + [i // 2 for i in range(20)], np.int32)]


@pytest.mark.parametrize("shape", ["small", "chain", "wide", "large"])
def test_waves_agree(shape):
    m = configs.random_trees(parents=_parents(shape), t_final_ms=4.0, seed=17, hh_everywhere=True)
    m.pulse_start = np.full(m.n_cells, 500.0, np.float32)
    res = {}
    for tpb, store in ((64, 1), (128, 1), (256, 1), (256, -1), (0, -1)):
        with Adjoint(m, checkpoint_steps=31, threads_per_cell=tpb, store_states=store) as adj:
            g0, a0 = adj.default_parameters()
            g = (g0 * 1.1).clone().requires_grad_(True)
            a = a0.clone().requires_grad_(True)
            target = adj.forward(g0, a0).clone()
            tr = trace(adj, g, a)
            ((tr - target) ** 2).mean().backward()
            res[tpb, store] = [x.detach().cpu().numpy() for x in (target, tr, g.grad, a.grad)]
    ref = oracle.run_f64_trace(m)
    first = res[64, 1]
    assert np.abs(first[0] - ref).max() < 1e-8
    assert np.isfinite(first[2]).all() and np.abs(first[2]).max() > 0
    for k, r in res.items():
        for x, y in zip(r, first):
            assert np.array_equal(x, y), k
