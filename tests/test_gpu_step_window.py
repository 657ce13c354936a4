"""Networks with multi-compartment cells, and of point neurons with generic synapses
(lems_window_kernel), several steps per launch (trig_fold_kernel): traces,
spikes, synaptic deliveries, last voltages and saved states equal the oracle's and those of
launches of one step, over delays around the shortest that allow a window and the longest window,
spikes that find one pending, odd chunks, other workgroup sizes, forced window lengths, captured graphs, and float times
whose step windows overlap (launches of one step)."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs, lems, lems_cells
from eden_amd.model import Model, Simulation
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
    ((3.0, 12.0), 25.0, {}), ((1.0, 4.0), 25.0, dict(size_limits=(256, 512, 1024, 2047))), ((1.0, 4.0), 23.7, {}), ((1.0, 4.0), 12.5, {})])
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


def _point_neurons(n, degree, delay_ms, seed, rings=0):
    """n Izhikevich and adaptive exponential cells, up to `degree` LEMS synapses each (some cells
    have none), then `rings` HH point cells without synapses."""
    rng = np.random.default_rng(seed)
    cells = lems_cells.build([
        ("izhikevich2007Cell", dict(v0=-60.0, C=100.0, k=0.7e-3, vr=-60.0, vt=-40.0, vpeak=35.0, a=0.03e-3, b=-2e-3,
                                    c=-50.0, d=0.1)),
        ("adExIaFCell", dict(C=281.0, gL=0.03, EL=-70.6, reset=-48.5, VT=-50.4, thresh=-40.4, refract=200.0, delT=2.0,
                             tauw=40000.0, a=4e-3, b=0.08))])
    types = lems.build([
        ("expTwoSynapse", dict(gbase=1e-3, erev=0.0, tauRise=500.0, tauDecay=5000.0), 1.0),
        ("alphaSynapse", dict(gbase=1e-3, erev=-80.0, tau=2000.0), 1.0)])
    hh = configs.hh_population(n_cells=rings, t_final_ms=30.0, seed=seed) if rings else None
    cnt = rng.integers(0, degree + 1, n)
    cnt[0], cnt[n // 2] = degree, 0
    begin = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    ns = int(begin[-1])
    pre = rng.integers(0, n, ns)
    order = np.argsort(pre, kind="stable")
    spikes = np.concatenate([[0], np.cumsum(np.bincount(pre, minlength=n))]).astype(np.int64)
    tail = lambda b, k: np.concatenate([b, np.full(k, b[-1])])
    full = lambda v, field: np.concatenate([v, getattr(hh, field)]) if rings else v
    nc = n + rings
    return Model(
        dt=25.0, t_final=30000.0, cell_comp_begin=np.arange(nc + 1), v0=full(np.zeros(n), "v0"),
        capacitance=full(np.ones(n), "capacitance"), area=full(np.ones(n), "area"), inv_rc_axial=np.zeros(nc),
        r_axial=np.zeros(nc), v_threshold=full(np.full(n, np.nan), "v_threshold"), parent=np.full(nc, -1),
        channel_types=hh.channel_types if rings else [],
        comp_chan_begin=full(np.zeros(n), "comp_chan_begin") if rings else np.zeros(n + 1),
        chan_type=hh.chan_type if rings else np.zeros(0), chan_gbase=hh.chan_gbase if rings else np.zeros(0),
        chan_erev=hh.chan_erev if rings else np.zeros(0), cell_rng_seed=configs.cell_rng_seeds(7, nc),
        comp_pulse_begin=np.arange(nc + 1), pulse_start=np.full(nc, 1000.0), pulse_duration=np.full(nc, 30000.0),
        pulse_amplitude=np.concatenate([rng.uniform(0.05, 0.9, n), np.full(rings, 0.1)]), pulse_weight=np.ones(nc),
        comp_syn_begin=tail(begin, rings),
        syn_type=np.concatenate([np.sort(rng.integers(0, 2, c)) for c in cnt] + [np.zeros(0, int)]),
        syn_weight=rng.uniform(0.5, 3.0, ns), syn_delay=np.round(rng.uniform(*delay_ms, ns) * 40.0) * 25.0,
        comp_spike_begin=tail(spikes, rings), spike_target=order, record_comp=np.arange(nc), event_comp=np.arange(nc),
        lems=types, lems_cells=cells, cell_lems_type=np.concatenate([rng.integers(0, 2, n), np.full(rings, -1)]),
        name="point_neurons")


@pytest.mark.parametrize("n,degree,delay_ms,rings,opt", [
    (1, 3, (1.0, 4.0), 0, {}), (15, 4, (0.1, 0.3), 0, {}), (16, 5, (0.05, 0.1), 0, {}), (17, 33, (1.0, 4.0), 0, dict(chunk_steps=37)),
    (40, 90, (0.5, 20.0), 0, dict(network_window=7)), (65, 12, (2.0, 6.0), 0, dict(use_graph=True, chunk_steps=300)),
    (33, 20, (1.0, 3.0), 5, {}), (20, 0, (1.0, 2.0), 0, {})])
def test_point_neuron_windows_equal_oracle_and_single_steps(n, degree, delay_ms, rings, opt):
    m = _point_neurons(n, degree, delay_ms, 3 + n, rings)
    tr, ev, syn, v, blob = _run(m, **opt)
    (ref, ec, er, _), (o_step, o_syn) = oracle.run_with_synapse_log(m)
    assert np.array_equal(tr, ref)
    assert len(er) > 0 or n == 1      # (the oracle's lone cell stays below its threshold)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
    assert np.array_equal(syn[0], o_step) and np.array_equal(syn[1], o_syn)
    t1, e1, s1, v1, b1 = _run(m, **{**opt, "network_window": -1, "use_graph": False})
    assert np.array_equal(t1, tr) and np.array_equal(v1, v) and np.array_equal(s1[0], syn[0])
    assert len(b1) == len(blob)
