"""Generic synapses of populations in which every cell has one instance or none (a lane a cell), two,
or a few, with cell counts around a wave, on physical point cells (launches of one step) and on
point neurons (windows of steps): traces, spikes and last voltages equal the oracle's."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs, lems, lems_cells
from eden_amd.model import Model, Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
TYPES = [("expTwoSynapse", dict(gbase=5e-3, erev=0.0, tauRise=500.0, tauDecay=5000.0), 1.0),
         ("alphaSynapse", dict(gbase=5e-3, erev=-80.0, tau=2000.0), 1.0)]


def _connections(n, most, rng):
    cnt = rng.integers(0, most + 1, n)
    cnt[0], cnt[-1] = most, most
    begin = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    ns = int(begin[-1])
    pre = rng.integers(0, n, ns)
    spikes = np.concatenate([[0], np.cumsum(np.bincount(pre, minlength=n))]).astype(np.int64)
    return dict(comp_syn_begin=begin, syn_type=np.concatenate([np.sort(rng.integers(0, 2, c)) for c in cnt]),
                syn_weight=rng.uniform(0.5, 3.0, ns), syn_delay=np.round(rng.uniform(0.5, 2.0, ns) * 40.0) * 25.0,
                comp_spike_begin=spikes, spike_target=np.argsort(pre, kind="stable"), lems=lems.build(TYPES))


def _physical(n, most, rng):
    m = configs.hh_population(n_cells=n, t_final_ms=10.0, seed=n, amp_max_nA=0.3)
    return dataclasses.replace(m, pulse_start=np.full(n, 500.0, np.float32), **_connections(n, most, rng))


def _neurons(n, most, rng):
    cells = lems_cells.build([("izhikevich2007Cell", dict(v0=-60.0, C=100.0, k=0.7e-3, vr=-60.0, vt=-40.0, vpeak=35.0,
                                                          a=0.03e-3, b=-2e-3, c=-50.0, d=0.1))])
    one = np.arange(n + 1)
    return Model(
        dt=25.0, t_final=20000.0, cell_comp_begin=one, v0=np.zeros(n), capacitance=np.ones(n), area=np.ones(n),
        inv_rc_axial=np.zeros(n), r_axial=np.zeros(n), v_threshold=np.full(n, np.nan), parent=np.full(n, -1),
        channel_types=[], comp_chan_begin=np.zeros(n + 1), chan_type=np.zeros(0), chan_gbase=np.zeros(0),
        chan_erev=np.zeros(0), cell_rng_seed=configs.cell_rng_seeds(7, n), comp_pulse_begin=one,
        pulse_start=np.full(n, 1000.0), pulse_duration=np.full(n, 30000.0), pulse_amplitude=rng.uniform(0.3, 0.9, n),
        pulse_weight=np.ones(n), record_comp=np.arange(n), event_comp=np.arange(n), lems_cells=cells,
        cell_lems_type=np.zeros(n, int), name="neurons", **_connections(n, most, rng))


@pytest.mark.parametrize("make", [_physical, _neurons])
@pytest.mark.parametrize("n,most", [(1, 1), (63, 1), (64, 1), (65, 1), (200, 1), (65, 2), (16, 3), (130, 4), (33, 5)])
def test_few_instances_a_cell(make, n, most):
    m = make(n, most, np.random.default_rng(10 * n + most))
    with Simulation(m, chunk_steps=53) as sim:
        tr, ev, v = sim.run_all(), sim.read_events(), sim.voltages()
    ref, ec, er, rv = oracle.run(m)
    assert len(er) > 0 or n == 1      # (a lone neuron stays below its threshold)
    assert np.array_equal(tr, ref) and np.array_equal(v, rv)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
