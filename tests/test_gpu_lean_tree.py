"""Cells of passive dendrites on an active soma (lean_tree_kernel): traces, spikes and last
voltages equal the oracle's bit for bit, and those of the general kernel on the same cells (which
a recorded dendrite selects), over sizes around the kernel's slots, every workgroup size with and
without a channel wave, lists of more rounds than headers are held, a root with more children than
a wave has lanes, and passive, unrecorded and several times stimulated roots."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
MS = 1000.0


def _parents(shape, n, rng):
    if shape == "chain":
        return np.arange(-1, n - 1, dtype=np.int32)
    if shape == "star":
        return np.concatenate([[-1], np.zeros(n - 1)]).astype(np.int32)
    if shape == "broom":                     # a chain to a fan
        return np.concatenate([np.arange(-1, n // 2), np.full(n - n // 2 - 1, n // 2)]).astype(np.int32)
    if shape == "wide":                      # few levels, many children a node
        return np.array([-1] + [int(rng.integers(max(1, i // 8))) for i in range(1, n)], np.int32)
    return np.array([-1] + [max(0, i - 1 - int(rng.integers(3))) for i in range(1, n)], np.int32)


def _model(shape, sizes, seed, passive_root=False):
    rng = np.random.default_rng(seed)
    m = configs.random_trees(parents=[_parents(shape, n, rng) for n in sizes], t_final_ms=6.0, seed=seed)
    roots = m.cell_comp_begin[:-1]
    nc, n = m.n_comps, len(sizes)
    # three overlapping pulses at every root, voltages of every compartment its own
    count = np.zeros(nc + 1, np.int64)
    count[roots + 1] = 3
    m = dataclasses.replace(
        m, v0=rng.uniform(-75.0, -55.0, nc).astype(np.float32), comp_pulse_begin=np.cumsum(count),
        pulse_start=np.tile(np.float32([0.3, 1.0, 2.5]) * MS, n), pulse_duration=np.full(3 * n, 2.0 * MS, np.float32),
        pulse_amplitude=rng.uniform(0.1, 0.5, 3 * n).astype(np.float32), pulse_weight=np.ones(3 * n, np.float32),
        record_comp=roots[: max(1, n - 1)].copy())       # the last root is not recorded
    if passive_root:
        b, t, g, e = configs._hh_channels(nc, np.zeros(nc, bool))
        m = dataclasses.replace(m, comp_chan_begin=b, chan_type=t, chan_gbase=g, chan_erev=e)
    return m


def _run(m, **opt):
    with Simulation(m, **opt) as sim:
        tr = sim.run_all()
        return tr, sim.read_events(), sim.voltages()


@pytest.mark.parametrize("shape,sizes,threads,wave", [
    ("chain", (2, 3, 64, 65, 128, 256), 64, 1), ("chain", (129, 257, 300, 512), 128, -1), ("chain", (513, 1024), 256, 1),
    ("chain", (1025, 1300, 2047), 512, 1), ("star", (3, 64, 65, 66, 129, 130, 200), 64, -1), ("star", (300, 511), 128, 1),
    ("star", (1200,), 0, 0), ("broom", (5, 100, 255, 256), 64, 1), ("broom", (400, 512), 128, 1), ("wide", (2, 9, 63, 192, 193, 250), 64, 1),
    ("wide", (511, 512), 128, -1), ("wide", (513, 1000), 256, -1), ("wide", (1023, 1500, 2000), 512, -1),
    ("narrow", (10, 40, 127, 128, 129, 250), 0, 0), ("narrow", (257, 640, 1024, 1800), 0, 0)])
@pytest.mark.parametrize("passive_root", [False, True])
def test_lean_trees_equal_oracle_and_general_kernel(shape, sizes, threads, wave, passive_root):
    m = _model(shape, sizes, 31 + len(sizes), passive_root)
    opt = dict(threads_per_cell=threads, channel_wave=(wave,) * 4)
    tr, ev, v = _run(m, chunk_steps=37, **opt)
    ref, ec, er, _ = oracle.run(m)
    assert np.array_equal(tr, ref), float(np.abs(tr - ref).max())
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
    general = dataclasses.replace(m, record_comp=np.concatenate([m.record_comp, m.cell_comp_begin[1:] - 1]))
    tg, eg, vg = _run(general, **opt)
    assert np.array_equal(tg[:, : tr.shape[1]], tr) and np.array_equal(vg, v)
    assert np.array_equal(eg[0], ev[0]) and np.array_equal(eg[1], ev[1])


def test_lean_trees_resume_from_a_saved_state():
    m = _model("narrow", (30, 200, 300, 700, 1500), 77)
    ref, _, v = _run(m)
    with Simulation(m) as a:
        a.run(100)
        blob = a.get_state()
    with Simulation(m) as b:
        b.set_state(blob)
        b.run_static()
        rows, row0 = b.read_trace()
        assert np.array_equal(rows, ref[row0:row0 + len(rows)]) and row0 + len(rows) == len(ref)
        assert np.array_equal(b.voltages(), v)
