"""The simulations whose speed is measured, each through the framework's public entry points
(`Simulation` for a model that runs forward, `adjoint.trace` for one that is fitted).

A pass of a forward case is what a program does with a model it holds: rewind it, run every
row, and read the recorded traces and the spike raster back. A pass of a fitting case is one
loss gradient: the differentiable forward run, a mean squared error against a target trace,
and the adjoint's backward run.

Sizes are those of the repository's configurations, scaled where a pass or its set-up would
take long, and of its tests. Trees of a population share a pool of morphologies, as the cells
of a NeuroML population share their cell type's, with densities and currents of their own.
"""
import dataclasses
import math

import numpy as np
import torch

from eden_amd import configs, lems, lems_cells
from eden_amd.adjoint import Adjoint, trace
from eden_amd.model import Model, Simulation, cell_rng_seeds

MS = 1000.0


def listed():
    return [
        # a handful of unconnected HH cells, as in the single-cell examples users start from:
        # the smallest call, bound by one cell's serial step
        dict(name="pop_24", kind="pop", cells=24, ms=10.0),
        # the 1,000-cell HH population, every cell recorded
        dict(name="pop_1000", kind="pop", cells=1000, ms=100.0),
        # a few reconstructed cells (active soma, passive dendrites) under current steps
        dict(name="trees_7", kind="trees", cells=7, lo=20, hi=300, pool=7, active=False, ms=25.0),
        # the 512-tree cable population: mid-sized cells, one wave each
        dict(name="trees_512", kind="trees", cells=512, lo=20, hi=400, pool=64, active=False, ms=50.0),
        # a population of very uneven cells, 10 to 2,000 compartments
        dict(name="trees_uneven", kind="trees", cells=2048, lo=10, hi=2000, pool=96, active=False, ms=25.0),
        # active dendrites: HH channels on every compartment
        dict(name="trees_active", kind="trees", cells=256, lo=60, hi=160, pool=64, active=True, ms=50.0),
        # a small recurrent network of HH point cells with Poisson drive
        dict(name="net_1000", kind="net", cells=1000, degree=50, ms=100.0),
        # a large one (in-degree 100 as in the 100,000-cell network)
        dict(name="net_24000", kind="net", cells=24000, degree=100, ms=50.0),
        # a network of multi-compartment and point cells, synapses on dendrites
        dict(name="mixed_48", kind="mixed", cells=48, points=150, conns=1500, ms=25.0),
        # artificial cells (Izhikevich, adaptive exponential) with LEMS synapses, generated code
        dict(name="lems_700", kind="lems", cells=700, degree=30, ms=50.0),
        # fitting a few small cells: a gradient of every channel density and current
        dict(name="adjoint_5", kind="adjoint", cells=5, comps=24, ms=10.0),
        # the fitting population, 100 compartments a cell, HH on every one
        dict(name="adjoint_256", kind="adjoint", cells=256, comps=100, ms=25.0),
    ]


def draw(rng):
    """One more case of the listed ones' ranges."""
    def log_int(a, b):
        return int(round(math.exp(rng.uniform(math.log(a), math.log(b)))))

    kind = rng.choice(["pop", "trees", "trees", "net", "mixed", "lems", "adjoint"])
    ms = round(rng.uniform(5.0, 40.0) / 0.025) * 0.025
    if kind == "pop":
        return dict(kind=kind, cells=log_int(1, 4000), ms=ms)
    if kind == "trees":
        active = rng.random() < 0.4
        hi = log_int(30, 300 if active else 2000)
        cells = max(1, min(log_int(1, 1500), int((20000 if active else 250000) / (0.4 * hi))))
        return dict(kind=kind, cells=cells, lo=max(2, int(hi * rng.uniform(0.02, 0.5))), hi=hi,
                    pool=min(cells, rng.randint(1, 64)), active=active, ms=min(ms, 20.0))
    if kind == "net":
        cells = log_int(60, 20000)
        return dict(kind=kind, cells=cells, degree=rng.randint(5, min(180, cells - 1)), ms=ms)
    if kind == "mixed":
        return dict(kind=kind, cells=log_int(2, 48), points=log_int(2, 150), conns=log_int(20, 1500), ms=min(ms, 20.0))
    if kind == "lems":
        cells = log_int(10, 700)
        return dict(kind=kind, cells=cells, degree=rng.randint(1, min(40, cells - 1)), ms=ms)
    return dict(kind=kind, cells=log_int(1, 256), comps=log_int(3, 110), ms=min(ms, 20.0))


# --------------------------------------------------------------------------- models


def _tree_population(case, seed):
    """`cells` trees of `lo` to `hi` compartments (log-uniform) over `pool` morphologies: HH on
    the soma or on every compartment, per-cell density factors U(0.5, 1.5), a somatic current
    step U(0.1, 0.5) nA from 2 ms on; somatic traces and spikes recorded."""
    rng = np.random.default_rng([4, seed])
    sizes = np.round(np.exp(rng.uniform(np.log(case["lo"]), np.log(case["hi"]), case["pool"]))).astype(np.int64)
    base = configs.random_trees(sizes=np.maximum(sizes, 2), t_final_ms=case["ms"], seed=rng.integers(1 << 30),
                                hh_everywhere=case["active"])
    pick = rng.integers(0, case["pool"], case["cells"])
    cb = base.cell_comp_begin
    n_of = (cb[1:] - cb[:-1])[pick]
    begin = np.concatenate([[0], np.cumsum(n_of)]).astype(np.int64)
    comp = np.concatenate([np.arange(cb[p], cb[p + 1]) for p in pick])
    cell_of = np.repeat(np.arange(case["cells"]), n_of)

    def spread(b):
        cnt = (b[1:] - b[:-1])[comp]
        nb = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
        return nb, np.repeat(b[:-1][comp] - nb[:-1], cnt) + np.arange(nb[-1])

    ch_b, ch = spread(base.comp_chan_begin)
    pu_b, pu = spread(base.comp_pulse_begin)
    factor = rng.uniform(0.5, 1.5, (case["cells"], 3)).astype(np.float32)
    factor[:, 0] = 1.0                       # the leak keeps its density
    chan_cell = np.repeat(cell_of, ch_b[1:] - ch_b[:-1])
    n = case["cells"]
    m = Model(
        dt=base.dt, t_final=base.t_final, cell_comp_begin=begin, v0=base.v0[comp], capacitance=base.capacitance[comp],
        area=base.area[comp], inv_rc_axial=base.inv_rc_axial[comp], r_axial=base.r_axial[comp],
        v_threshold=base.v_threshold[comp], parent=base.parent[comp], channel_types=base.channel_types,
        comp_chan_begin=ch_b, chan_type=base.chan_type[ch],
        chan_gbase=base.chan_gbase[ch] * factor[chan_cell, base.chan_type[ch]], chan_erev=base.chan_erev[ch],
        cell_rng_seed=cell_rng_seeds(1, n), comp_pulse_begin=pu_b, pulse_start=np.full(len(pu), 2.0 * MS),
        pulse_duration=np.full(len(pu), case["ms"] * MS), pulse_amplitude=rng.uniform(0.1, 0.5, len(pu)),
        pulse_weight=np.ones(len(pu)), record_comp=begin[:-1].copy(), event_comp=begin[:-1].copy(), name="trees")
    return m


def _population(case, seed):
    m = configs.hh_population(n_cells=case["cells"], t_final_ms=case["ms"], seed=10 + seed)
    return dataclasses.replace(m, pulse_start=np.full(case["cells"], min(10.0, 0.2 * case["ms"]) * MS, np.float32))


def _lems_network(case, seed):
    """Izhikevich (2007) and adaptive exponential cells, `degree` connections onto each, LEMS
    synapses of two types, a current step into every cell."""
    rng = np.random.default_rng([9, seed])
    n, k = case["cells"], case["degree"]
    cells = lems_cells.build([
        ("izhikevich2007Cell", dict(v0=-60.0, C=100.0, k=0.7e-3, vr=-60.0, vt=-40.0, vpeak=35.0, a=0.03e-3, b=-2e-3,
                                    c=-50.0, d=0.1)),
        ("adExIaFCell", dict(C=281.0, gL=0.03, EL=-70.6, reset=-48.5, VT=-50.4, thresh=-40.4, refract=200.0, delT=2.0,
                             tauw=40000.0, a=4e-3, b=0.08))])
    types = lems.build([
        ("expTwoSynapse", dict(gbase=1e-3, erev=0.0, tauRise=500.0, tauDecay=5000.0), 1.0),
        ("alphaSynapse", dict(gbase=1e-3, erev=-80.0, tau=2000.0), 1.0)])
    ctype = (rng.random(n) < 0.3).astype(np.int32)
    pre = np.argsort(rng.random((n, n)), axis=1)[:, :k] if n <= 64 else rng.integers(0, n, (n, k))
    inhibitory = np.sort(rng.random((n, k)) < 0.2, axis=1)
    begin = np.arange(n + 1, dtype=np.int64)
    order = np.argsort(pre.ravel(), kind="stable")
    spikes = np.concatenate([[0], np.cumsum(np.bincount(pre.ravel(), minlength=n))]).astype(np.int64)
    return Model(
        dt=25.0, t_final=case["ms"] * MS, cell_comp_begin=begin, v0=np.zeros(n), capacitance=np.ones(n),
        area=np.ones(n), inv_rc_axial=np.zeros(n), r_axial=np.zeros(n), v_threshold=np.full(n, np.nan),
        parent=np.full(n, -1), channel_types=[], comp_chan_begin=np.zeros(n + 1), chan_type=np.zeros(0),
        chan_gbase=np.zeros(0), chan_erev=np.zeros(0), cell_rng_seed=cell_rng_seeds(7, n),
        comp_pulse_begin=begin, pulse_start=np.full(n, 1.0 * MS), pulse_duration=np.full(n, case["ms"] * MS),
        pulse_amplitude=rng.uniform(0.05, 0.9, n), pulse_weight=np.ones(n),
        comp_syn_begin=begin * k, syn_type=inhibitory.astype(np.int32).ravel(),
        syn_weight=rng.uniform(0.5, 3.0, n * k), syn_delay=np.round(rng.uniform(1.0, 4.0, n * k) * MS / 25.0) * 25.0,
        comp_spike_begin=spikes, spike_target=order, record_comp=np.arange(min(n, 64)), event_comp=np.arange(n),
        lems=types, lems_cells=cells, cell_lems_type=ctype, name="lems_network")


def _model(case, seed):
    kind = case["kind"]
    if kind == "pop":
        return _population(case, seed)
    if kind == "trees":
        return _tree_population(case, seed)
    if kind == "net":
        return configs.spiking_network(n_cells=case["cells"], in_degree=case["degree"], t_final_ms=case["ms"],
                                       seed=30 + seed, sim_seed=3 + seed, poisson_hz=40.0)
    if kind == "mixed":
        rng = np.random.default_rng([7, seed])
        sizes = np.round(np.exp(rng.uniform(np.log(20), np.log(400), case["cells"]))).astype(int)
        return configs.mixed_network(tree_sizes=tuple(int(s) for s in sizes), n_point=case["points"],
                                     n_conn=case["conns"], t_final_ms=case["ms"], seed=50 + seed, sim_seed=5 + seed)
    if kind == "lems":
        return _lems_network(case, seed)
    m, g0 = configs.config5(n_cells=case["cells"], n_comps=case["comps"], t_final_ms=case["ms"], seed=60 + seed,
                            init_seed=70 + seed)
    m = dataclasses.replace(m, pulse_start=np.full(case["cells"], 1.0 * MS, np.float32))
    return m, g0


# --------------------------------------------------------------------------- passes


def prepare(case, seed):
    if case["kind"] == "adjoint":
        m, g0 = _model(case, seed)
        adj = Adjoint(m)
        g_true, a = adj.default_parameters()
        target = adj.forward(g_true, a).clone()
        return dict(adj=adj, target=target, gbase=torch.tensor(g0, dtype=torch.float64, device=adj.device,
                                                               requires_grad=True), amp=a.clone().requires_grad_(True))
    m = _model(case, seed)
    # room for 500 spikes a second and cell; networks record some cells only, so their
    # programs also look at every cell's last voltage
    return dict(sim=Simulation(m), spikes=(2, m.n_cells * (1 + int(case["ms"] / 2))),
                all_recorded=case["kind"] not in ("net", "lems"))


def run(state):
    if "adj" in state:
        v = trace(state["adj"], state["gbase"], state["amp"])
        loss = ((v - state["target"]) ** 2).sum() / v.numel()
        g, a = torch.autograd.grad(loss, (state["gbase"], state["amp"]))
        return dict(trace=v.detach(), grad_gbase=g, grad_amplitude=a)
    sim = state["sim"]
    sim.reset()
    v = sim.run_all()
    col, row = sim.read_events()
    spikes = np.full(state["spikes"], -1, np.int64)     # (column, row) of each, -1 past the last
    spikes[0, :len(col)], spikes[1, :len(row)] = col, row
    if not state["all_recorded"]:
        return dict(trace=v, spikes=spikes, final=sim.voltages())
    return dict(trace=v, spikes=spikes)


def _rows(case):
    return int(case["ms"] * MS / 25.0 + 1e-9) + 1


def work(case):
    """Bytes and operations of one pass. A model's state can stay on the chip for the run, so
    the bytes are its tables once and its recorded rows once (about 60 a compartment, 30 a
    synapse). Operations: about 150 a gate variable and step (two rates of one exponential each
    and the update), 30 a compartment and step (currents, membrane update, elimination and
    substitution), 20 a synapse and step; a gradient costs three forward passes."""
    rows, kind, n = _rows(case), case["kind"], case["cells"]
    gate, comp_ops, syn_ops = 150.0, 30.0, 20.0
    if kind == "pop":
        return dict(bytes=n * (100.0 + 4.0 * rows), flops=rows * n * (3 * gate + comp_ops))
    if kind == "trees":
        lo, hi = max(2, case["lo"]), case["hi"]
        comps = n * ((hi - lo) / math.log(hi / lo) if hi > lo else hi)
        gates = 3 * comps if case["active"] else 3 * n
        return dict(bytes=comps * 60.0 + 4.0 * n * rows, flops=rows * (gates * gate + comps * comp_ops))
    if kind == "net":
        syn = n * case["degree"]
        return dict(bytes=n * 100.0 + syn * 30.0 + 4.0 * rows * min(n, 100),
                    flops=rows * (syn * syn_ops + n * (3 * gate + comp_ops)))
    if kind == "mixed":
        comps = n * 127.0
        return dict(bytes=(comps + case["points"]) * 60.0 + 4.0 * rows * (n + case["points"] + 8),
                    flops=rows * ((n + case["points"]) * 3 * gate + comps * comp_ops + case["conns"] * syn_ops))
    if kind == "lems":
        return dict(bytes=n * (100.0 + 30.0 * case["degree"]) + 4.0 * rows * min(n, 64),
                    flops=rows * n * (40.0 + case["degree"] * syn_ops))
    comps = n * case["comps"]
    return dict(bytes=comps * 100.0 + 8.0 * 3 * rows * n, flops=3.0 * rows * comps * (3 * gate + comp_ops))


# --------------------------------------------------------------------------- 64 bits


_HH_RATES = [float(np.float32(r / 1e3)) for r in (1.0, 4.0, 0.07, 1.0, 0.1, 0.125)]
_QMIN, _QMAX = float(np.float32(1e-6)), 1.0 - float(np.float32(1e-6))


def _hh_rates(V, xp):
    def lin(r, mid, sc):
        x = (V - mid) / sc
        safe = xp.where(x == 0, xp.ones_like(x), x)
        return r * xp.where(x == 0, xp.ones_like(x), safe / (1.0 - xp.exp(-safe)))

    r = _HH_RATES                            # the model's fp32 parameters
    return ((lin(r[0], -40.0, 10.0), r[1] * xp.exp((V + 65.0) / -18.0)),
            (r[2] * xp.exp((V + 65.0) / -20.0), r[3] / (1.0 + xp.exp((-35.0 - V) / 10.0))),
            (lin(r[4], -55.0, 10.0), r[5] * xp.exp((V + 65.0) / -80.0)))


def _hh_constants(m):
    """Per compartment leak, Na and K density (0 where absent) in 64 bits."""
    g = np.zeros((m.n_comps, 3))
    owner = np.repeat(np.arange(m.n_comps), np.diff(m.comp_chan_begin))
    g[owner, m.chan_type] = m.chan_gbase.astype(np.float64)
    return g


def _cable_levels(m):
    """Depth levels of the whole population's trees: (compartments, their parents) per depth."""
    start = np.repeat(m.cell_comp_begin[:-1], np.diff(m.cell_comp_begin))
    up = np.where(m.parent >= 0, m.parent + start, -1)
    depth = np.zeros(m.n_comps, np.int64)
    for c in np.flatnonzero(up >= 0):
        depth[c] = depth[up[c]] + 1
    return [(c, up[c]) for c in (np.flatnonzero(depth == d) for d in range(1, depth.max() + 1))]


def _forward64(m):
    """Recorded voltages of unconnected HH cells or trees in 64 bits (numpy): exponential-Euler
    gates, semi-implicit membrane, tree elimination and substitution over depth levels."""
    dt, rows = float(m.dt), int(m.t_final / float(m.dt) + 1e-9) + 1
    E = (-54.387, 50.0, -77.0)
    E = [float(np.float32(e)) for e in E]
    g, A = _hh_constants(m), m.area.astype(np.float64) * float(np.float32(1e-5))
    C, inv, V = m.capacitance.astype(np.float64), m.inv_rc_axial.astype(np.float64), m.v0.astype(np.float64)
    gated = np.flatnonzero(g[:, 1] > 0)
    ga = g[gated] * A[gated, None]
    leak = g[:, 0] * A
    q = [a / (a + b) for a, b in _hh_rates(V[gated], np)]
    levels = _cable_levels(m) if (m.parent >= 0).any() else []
    ui = [-dt / (m.r_axial[c].astype(np.float64) * C[c]) for c, _ in levels]
    uj = [-dt / (m.r_axial[c].astype(np.float64) * C[p]) for c, p in levels]
    at = np.repeat(np.arange(m.n_comps), np.diff(m.comp_pulse_begin))
    t0, t1 = m.pulse_start.astype(np.float64), (m.pulse_start + m.pulse_duration).astype(np.float64)
    amp = m.pulse_amplitude.astype(np.float64) * m.pulse_weight
    out = np.empty((rows, len(m.record_comp)))
    for r in range(rows):
        out[r] = V[m.record_comp]
        t = r * dt
        G = leak.copy()
        I = leak * (E[0] - V)
        na, kk = ga[:, 1] * q[0] ** 3 * q[1], ga[:, 2] * q[2] ** 4
        Vg = V[gated]
        G[gated] += na + kk
        I[gated] += na * (E[1] - Vg) + kk * (E[2] - Vg)
        np.add.at(I, at, np.where((t0 <= t) & (t <= t1), amp, 0.0))
        for s, (a, b) in enumerate(_hh_rates(Vg, np)):
            blend = np.exp(-dt * (a + b))
            q[s] = np.clip(blend * q[s] + (1.0 - blend) * a / (a + b), _QMIN, _QMAX)
        x = V + dt * (I + V * G) / C
        D = 1.0 + dt * (G / C + inv)
        for (c, p), i, j in zip(reversed(levels), reversed(ui), reversed(uj)):
            ratio = j / D[c]
            np.subtract.at(D, p, ratio * i)
            np.subtract.at(x, p, ratio * x[c])
        root = m.cell_comp_begin[:-1]
        x[root] /= D[root]
        for (c, p), i in zip(levels, ui):
            x[c] = (x[c] - i * x[p]) / D[c]
        V = x
    return out


def _gradient64(case, seed):
    """Trace and gradients of the fitting loss in 64 bits: torch on the CPU, one dense solve a
    step and cell, differentiated by autograd."""
    m, g0 = _model(case, seed)
    dt, rows, n, k = float(m.dt), _rows(case), case["cells"], case["comps"]
    f = lambda x: torch.tensor(np.asarray(x, np.float64).reshape(n, k))
    C, A, inv = f(m.capacitance), f(m.area) * float(np.float32(1e-5)), f(m.inv_rc_axial)
    E = [float(np.float32(e)) for e in (-54.387, 50.0, -77.0)]
    parent = m.parent.reshape(n, k)
    off = torch.zeros(n, k, k, dtype=torch.float64)
    for c in range(n):
        for i in range(1, k):
            p, R = parent[c, i], float(m.r_axial[c * k + i])
            off[c, i, p] = -dt / (R * float(C[c, i]))
            off[c, p, i] = -dt / (R * float(C[c, p]))
    t0, t1 = m.pulse_start.astype(np.float64), m.pulse_start.astype(np.float64) + m.pulse_duration

    def simulate(gbase, amp):
        g = gbase.reshape(n, k, 3)               # leak, Na, K on every compartment
        V = f(m.v0)
        q = [a / (a + b) for a, b in _hh_rates(V, torch)]
        out = []
        for r in range(rows):
            out.append(V[:, 0])
            gl, na, kk = g[..., 0] * A, g[..., 1] * A * q[0] ** 3 * q[1], g[..., 2] * A * q[2] ** 4
            G = gl + na + kk
            I = gl * (E[0] - V) + na * (E[1] - V) + kk * (E[2] - V)
            on = torch.tensor(((t0 <= r * dt) & (r * dt <= t1)) * m.pulse_weight.astype(np.float64))
            I = torch.cat([I[:, :1] + (amp * on)[:, None], I[:, 1:]], 1)
            nq = []
            for s, (a, b) in enumerate(_hh_rates(V, torch)):
                blend = torch.exp(-dt * (a + b))
                nq.append(torch.clamp(blend * q[s] + (1.0 - blend) * a / (a + b), _QMIN, _QMAX))
            D = 1.0 + dt * (G / C + inv)
            V = torch.linalg.solve(off + torch.diag_embed(D), (V + dt * (I + V * G) / C).unsqueeze(-1)).squeeze(-1)
            q = nq
        return torch.stack(out)

    amp = torch.tensor(m.pulse_amplitude.astype(np.float64), requires_grad=True)
    with torch.no_grad():
        target = simulate(torch.tensor(m.chan_gbase.astype(np.float64)), amp)
    gbase = torch.tensor(np.asarray(g0, np.float64), requires_grad=True)
    v = simulate(gbase, amp)
    gg, ga = torch.autograd.grad(((v - target) ** 2).sum() / v.numel(), (gbase, amp))
    return dict(trace=v.detach(), grad_gbase=gg, grad_amplitude=ga)


def exact(case, seed):
    """64-bit values for the cells that do not hear each other. Networks give none: which step
    an event falls into is decided by comparisons of the step's own arithmetic, so another
    precision's network is another trajectory. Large trees and fits would take too long."""
    rows = _rows(case)
    if case["kind"] == "pop" or (case["kind"] == "trees" and
                                 case["cells"] * case["hi"] * rows * (3 if case["active"] else 1) < 5e8):
        return dict(trace=_forward64(_model(case, seed)), spikes=None)
    if case["kind"] == "adjoint" and case["cells"] * case["comps"] ** 2 * rows < 5e6:
        return _gradient64(case, seed)
    return None
