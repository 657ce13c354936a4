"""Networks of tree cells and of point neurons: network_stats says how many steps a launch runs and
how many such windows ran, so that a model that should run windows is seen to; one step a launch
where a delay is too short, float step windows overlap, or generic synapses reach physical cells.
States saved after windows are those of launches of one step, byte for byte, and every last
voltage is the oracle's."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs, lems
from eden_amd.model import Simulation
from oracle import oracle
from tests.test_gpu_step_window import _model, _point_neurons

pytestmark = pytest.mark.gpu


def _ceil(a, b):      # (a run of that many rows takes as many steps after the initial ones)
    return -(-a // b)


def _run(m, **opt):
    with Simulation(m, **opt) as sim:
        sim.run_all()
        return sim.network_stats(), sim.voltages(), sim.get_state(), sim.total_rows


@pytest.mark.parametrize("delay_ms,dt,opt,steps", [
    ((0.075, 0.2), 25.0, {}, 1), ((0.1, 0.2), 25.0, {}, 2), ((0.5, 2.0), 25.0, {}, 18), ((3.0, 9.0), 25.0, {}, 64),
    ((1.0, 4.0), 25.0, dict(network_window=5), 5), ((1.0, 4.0), 25.0, dict(network_window=-1), 1),
    ((1.0, 4.0), 25.0, dict(use_graph=True), 38), ((1.0, 4.0), 23.7, {}, 1), ((1.0, 4.0), 25.0, dict(chunk_steps=101), 38)])
def test_trees(delay_ms, dt, opt, steps):
    m = _model(delay_ms, 21, dt)
    d = m.syn_delay.copy()
    d[m.spike_target[0]] = round(delay_ms[0] * 40.0) * 25.0      # the shortest delay is there
    m = dataclasses.replace(m, syn_delay=d)
    stats, v, blob, rows = _run(m, **opt)
    assert stats[0] == steps and stats[2] == 0 and stats[3] == -1
    if steps == 1:
        assert stats[1] == 0
    elif not opt:
        assert stats[1] == _ceil(rows, steps)
    else:
        assert stats[1] >= _ceil(rows, steps)
    assert np.array_equal(v, oracle.run(m)[3])
    single, v1, blob1, _ = _run(m, **{**opt, "network_window": -1, "use_graph": False})
    assert single[:2] == (1, 0)
    assert np.array_equal(v1, v) and blob1 == blob


@pytest.mark.parametrize("n,degree,delay_ms,rings,steps", [(40, 12, (0.5, 3.0), 0, 18), (33, 20, (2.0, 3.0), 5, 64), (17, 5, (0.05, 0.1), 0, 1)])
def test_point_neurons(n, degree, delay_ms, rings, steps):
    m = _point_neurons(n, degree, delay_ms, 3 + n, rings)
    d = m.syn_delay.copy()
    d[m.spike_target[0]] = round(delay_ms[0] * 40.0) * 25.0
    m = dataclasses.replace(m, syn_delay=d)
    with Simulation(m, log_synapse_events=1 << 20) as a, Simulation(m, log_synapse_events=1 << 20, network_window=-1) as b:
        assert np.array_equal(a.run_all(), b.run_all())
        assert a.network_stats()[0] == steps and b.network_stats()[:2] == (1, 0)
        assert (a.network_stats()[1] > 0) == (steps > 1)
        for x, y in zip(a.read_synapse_events(), b.read_synapse_events()):
            assert np.array_equal(x, y)
        assert np.array_equal(a.voltages(), b.voltages()) and a.get_state() == b.get_state()


def test_generic_synapses_on_physical_cells_run_single_steps():
    m = configs.mixed_network(tree_sizes=(20, 70), n_point=3, n_conn=40, t_final_ms=3.0)
    types = [("expTwoSynapse", dict(gbase=g, erev=e, tauRise=500.0, tauDecay=5000.0), 1.0) for g, e in ((2e-3, 0.0), (4e-3, -80.0))]
    m = dataclasses.replace(m, lems=lems.build(types), syn_types=[])
    assert _run(m)[0][:2] == (1, 0)
