"""Channels whose open fraction is a product of more than four gate factors: HH cells with m^5 h^2
and n^7 (and n alone, n^4, and a gate to the power 9 beside a channel of one) on point cells, in a
network of point cells, on the active root of a passive tree, on every compartment, and on fitted
cells. Forward runs equal the oracle's bit for bit; the fitted cells' gradient equals central
differences of the forward run as closely as HH cells' do."""
import dataclasses

import numpy as np
import pytest
import torch

from eden_amd import _native as N
from eden_amd import configs
from eden_amd.adjoint import Adjoint, trace
from eden_amd.model import Simulation, channel_type, rate
from oracle import oracle

pytestmark = pytest.mark.gpu


def _types(m_power, h_power, n_power):
    return [
        channel_type([]),
        channel_type([(m_power, rate(N.RATE_EXPLINEAR, 1.0, -40.0, 10.0), rate(N.RATE_EXP, 4.0, -65.0, -18.0)),
                      (h_power, rate(N.RATE_EXP, 0.07, -65.0, -20.0), rate(N.RATE_SIGMOID, 1.0, -35.0, 10.0))]),
        channel_type([(n_power, rate(N.RATE_EXPLINEAR, 0.1, -55.0, 10.0), rate(N.RATE_EXP, 0.125, -65.0, -80.0))])]


POWERS = [(5, 2, 7), (3, 2, 4), (4, 1, 1), (1, 9, 5)]


def _with(m, powers):
    return dataclasses.replace(m, channel_types=_types(*powers), pulse_start=np.full(len(m.pulse_start), 500.0, np.float32))


def _check(m, kernel):
    with Simulation(m, chunk_steps=77) as sim:
        tr, ev, v = sim.run_all(), sim.read_events(), sim.voltages()
        assert kernel in {k["symbol"].split("<")[0] for k in sim.kernel_infos()}
    ref, ec, er, rv = oracle.run(m)
    assert ref.max() - ref.min() > 5.0
    assert np.array_equal(tr, ref) and np.array_equal(v, rv)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)


@pytest.mark.parametrize("powers", POWERS)
def test_forward_equals_oracle(powers):
    _check(_with(configs.hh_population(n_cells=21, t_final_ms=20.0, amp_max_nA=0.5), powers), "point_quad_kernel")
    net = configs.spiking_network(n_cells=37, in_degree=20, t_final_ms=20.0, poisson_hz=300.0, weight_mu=2.0)
    _check(_with(net, powers), "net_quad_kernel")
    sizes = [20, 130, 300, 1200]
    _check(_with(configs.random_trees(sizes=sizes, n_cells=4, t_final_ms=15.0, seed=3), powers), "lean_tree_kernel")
    _check(_with(configs.random_trees(sizes=sizes, n_cells=4, t_final_ms=8.0, seed=3, hh_everywhere=True), powers), "tree_kernel")
    mixed = configs.mixed_network(tree_sizes=(20, 90), n_point=9, n_conn=80, t_final_ms=15.0)
    _check(_with(mixed, powers), "point_kernel")


@pytest.mark.parametrize("powers", POWERS)
def test_gradient_equals_central_differences(powers):
    m, g0 = configs.config5(n_cells=2, n_comps=12, t_final_ms=8.0)
    m = _with(m, powers)
    res = {}
    for threads in (64, 128, 256):
        with Adjoint(m, checkpoint_steps=37, threads_per_cell=threads) as adj:
            gt, a0 = adj.default_parameters()
            target = adj.forward(gt, a0).clone()
            assert np.abs(target.cpu().numpy() - oracle.run_f64_trace(m)).max() < 1e-8
            g = torch.tensor(g0, dtype=torch.float64, device=gt.device, requires_grad=True)
            a = (a0 * 1.05).clone().requires_grad_(True)
            loss = lambda x, y: ((adj.forward(x, y) - target) ** 2).sum() / target.numel()
            L = ((trace(adj, g, a) - target) ** 2).sum() / target.numel()
            L.backward()
            res[threads] = (g.grad.cpu().numpy(), a.grad.cpu().numpy())
            if threads != 128:
                continue
            base = g.detach()
            scale = float(g.grad.abs().max())
            for k in np.argsort(-(g.grad * base).abs().cpu().numpy())[:6]:
                h = 1e-6 * float(base[k])
                up, down = base.clone(), base.clone()
                up[k] += h
                down[k] -= h
                fd = float(loss(up, a.detach()) - loss(down, a.detach())) / float(up[k] - down[k])
                assert abs(fd - float(g.grad[k])) <= 1e-4 * abs(fd) + 1e-9 * scale, (k, fd, float(g.grad[k]))
    for r in res.values():
        for x, y in zip(r, res[64]):
            assert np.isfinite(x).all() and np.array_equal(x, y)
