"""Networks with multi-compartment cells, several steps per launch (trig_fold_kernel): traces,
spikes, synaptic deliveries, last voltages and saved states equal the oracle's and those of
launches of one step, over delays around the shortest that allow a window and the longest window,
spikes that find one pending, odd chunks, forced window lengths, captured graphs, and float times
whose step windows overlap (launches of one step)."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu


def _model(delay_ms, seed, dt=25.0):
    m = configs.mixed_network(tree_sizes=(20, 70, 140, 300), n_point=20, n_conn=300, t_final_ms=30.0, seed=seed,
                              delay_ms=delay_ms, weight=(3.0, 9.0), amp_range=(0.5, 0.9))
    return dataclasses.replace(m, dt=dt, pulse_start=np.full(len(m.pulse_start), 500.0, np.float32))


def _run(m, **opt):
    with Simulation(m, log_synapse_events=1 << 20, **opt) as sim:
        tr = sim.run_all()
        return tr, sim.read_events(), sim.read_synapse_events(), sim.voltages(), sim.get_state()


@pytest.mark.parametrize("delay_ms,dt,opt", [
    ((0.05, 0.1), 25.0, {}), ((0.1, 0.2), 25.0, {}), ((0.1, 30.0), 25.0, dict(chunk_steps=37)),
    ((1.0, 4.0), 25.0, {}), ((1.0, 4.0), 25.0, dict(network_window=5, chunk_steps=101)),
    ((1.0, 4.0), 25.0, dict(use_graph=True, chunk_steps=300)), ((1.7, 20.0), 25.0, dict(chunk_steps=1)),
    ((3.0, 12.0), 25.0, {}), ((1.0, 4.0), 23.7, {}), ((1.0, 4.0), 12.5, {})])
def test_windows_equal_oracle_and_single_steps(delay_ms, dt, opt):
    m = _model(delay_ms, 21, dt)
    tr, ev, syn, v, blob = _run(m, **opt)
    (ref, ec, er, _), (o_step, o_syn) = oracle.run_with_synapse_log(m)
    assert len(o_step) > 100
    assert np.array_equal(tr, ref), float(np.abs(tr - ref).max())
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
    assert np.array_equal(syn[0], o_step) and np.array_equal(syn[1], o_syn)
    t1, e1, s1, v1, b1 = _run(m, **{**opt, "network_window": -1, "use_graph": False})
    assert np.array_equal(t1, tr) and np.array_equal(v1, v)
    assert len(b1) == len(blob)


def test_state_saved_by_windows_resumes_in_single_steps():
    m = _model((1.0, 9.0), 5)
    ref = _run(m)[0]
    for save, resume in ((0, -1), (-1, 0)):
        with Simulation(m, network_window=save, chunk_steps=613) as a:
            a.run(613)
            blob = a.get_state()
        with Simulation(m, network_window=resume, chunk_steps=613) as b:
            b.set_state(blob)
            b.run_static()
            rows, row0 = b.read_trace()
            assert row0 >= 612 and len(rows) > 500
            assert np.array_equal(rows, ref[row0:row0 + len(rows)])
