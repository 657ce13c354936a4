"""Workgroup sizes of a network's tree cells: small cells get more lanes where launches run several
steps, and share few sizes where every launch is of one step (delays of a step or two, launches of
one step asked for, generic synapses); traces equal the oracle's with both."""
import dataclasses

import numpy as np
import pytest

from eden_amd import autotune, configs, lems
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
SIZES = (40, 64, 65, 100, 129, 250, 300, 513, 1100)
WINDOW, SINGLE = (64, 128, 512, 2047), (256, 512, 512, 2047)


def _sizes(limits):
    return sorted(next(t for t, l in zip((64, 128, 256, 512), limits) if n <= l) for n in SIZES)


def _generic(m):
    types = [("expTwoSynapse", dict(gbase=g, erev=e, tauRise=500.0, tauDecay=5000.0), 1.0) for g, e in ((2e-3, 0.0), (4e-3, -80.0))]
    return dataclasses.replace(m, lems=lems.build(types), syn_types=[])


@pytest.mark.parametrize("delay_ms,generic,opt,limits", [
    ((1.0, 4.0), False, {}, WINDOW), ((0.1, 0.2), False, {}, WINDOW), ((0.075, 0.2), False, {}, SINGLE),
    ((0.025, 0.05), False, {}, SINGLE), ((1.0, 4.0), False, dict(network_window=-1), SINGLE), ((1.0, 4.0), True, {}, SINGLE)])
def test_sizes_follow_the_steps_per_launch(delay_ms, generic, opt, limits):
    m = configs.mixed_network(tree_sizes=SIZES, n_point=6, n_conn=150, t_final_ms=6.0, seed=8, delay_ms=delay_ms,
                              weight=(3.0, 9.0))
    m = dataclasses.replace(m, pulse_start=np.full(len(m.pulse_start), 300.0, np.float32))
    if generic:
        m = _generic(m)
    with Simulation(m, **opt) as sim:
        tr, ev, v = sim.run_all(), sim.read_events(), sim.voltages()
        infos = [k for k in sim.kernel_infos() if k["comps"] > k["cells"]]
    assert sorted(k["threads_per_block"] for k in infos for _ in range(k["cells"])) == _sizes(limits)
    ref, ec, er, rv = oracle.run(m)
    assert len(er) > 0
    assert np.array_equal(tr, ref) and np.array_equal(v, rv)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)


def test_autotuner_starts_from_the_networks_limits():
    m = configs.mixed_network(tree_sizes=SIZES, n_point=6, n_conn=150, t_final_ms=5.0, seed=8)
    assert autotune.size_rule(m) == (WINDOW, autotune.NETWORK_CANDIDATES)
    limits, report = autotune.autotune(m, steps=60, repeats=1)
    print(f"[autotune] {limits} from {report}", flush=True)
    times = dict(report)
    assert report[0][0] == WINDOW and times[limits] <= times[WINDOW]
    with Simulation(m) as a, Simulation(m, size_limits=limits) as b:
        assert a.size_limits() == WINDOW and b.size_limits() == limits
        assert np.array_equal(a.run_all(), b.run_all())


@pytest.mark.parametrize("largest,limits", [(1024, (256, 512, 1024, 2047)), (1025, SINGLE)])
def test_single_steps_share_the_largest_size_where_a_cell_needs_it(largest, limits):
    m = configs.mixed_network(tree_sizes=(40, 600, largest), n_point=2, n_conn=30, t_final_ms=2.0, delay_ms=(0.025, 0.05))
    with Simulation(m) as sim:
        assert sim.size_limits() == limits
        tr = sim.run_all()
    assert np.array_equal(tr, oracle.run(m)[0])
