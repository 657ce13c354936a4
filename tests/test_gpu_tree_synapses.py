"""Synapse lists of tree compartments around the numbers the kernels read at a time (two, or eight
where a compartment has a long list): several types in a list, somata and dendrites, launches of
one step and of several; traces, spikes, every delivery and the last voltages equal the oracle's."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
MS = 1000.0


def _network(sizes, counts, delay_ms, seed):
    """Tree cells of `sizes`; cell c's soma gets counts[c] synapses, two of its dendrites
    counts[c - 1] and one."""
    rng = np.random.default_rng(seed)
    m = configs.mixed_network(tree_sizes=sizes, n_point=6, n_conn=10, t_final_ms=8.0, seed=seed, amp_range=(0.5, 0.9))
    begin, nc = m.cell_comp_begin, m.n_comps
    somata = begin[:-1]
    tgt = []
    for c in range(len(sizes)):
        tgt += [begin[c]] * counts[c] + [begin[c] + 1] * counts[c - 1] + [begin[c + 1] - 1]
    tgt = np.array(tgt, np.int64)
    n = len(tgt)
    src = somata[rng.integers(0, len(somata), n)]
    stype = rng.integers(0, 2, n).astype(np.int32)
    order = np.lexsort((np.arange(n), stype, tgt))
    inst = np.empty(n, np.int64)
    inst[order] = np.arange(n)
    by_src = np.argsort(src, kind="stable")
    csr = lambda at: np.concatenate([[0], np.cumsum(np.bincount(at, minlength=nc))]).astype(np.int64)
    return dataclasses.replace(
        m, pulse_start=np.full(len(m.pulse_start), 300.0, np.float32), comp_syn_begin=csr(tgt), syn_type=stype[order],
        syn_weight=rng.uniform(0.3, 1.5, n).astype(np.float32), comp_spike_begin=csr(src), spike_target=inst[by_src],
        syn_delay=(np.round(rng.uniform(*delay_ms, n) * MS / 25.0) * 25.0).astype(np.float32))


@pytest.mark.parametrize("delay_ms,opt", [((0.5, 2.0), {}), ((0.025, 0.1), {}), ((0.5, 2.0), dict(chunk_steps=41, network_window=3))])
@pytest.mark.parametrize("sizes,counts", [
    ((30, 60, 90, 120), (0, 1, 2, 3)), ((30, 60, 90, 120), (7, 8, 9, 15)), ((30, 70, 140, 600), (16, 17, 2, 1)),
    ((30, 70, 140, 600), (15, 33, 64, 130))])
def test_synapse_lists_of_tree_compartments(sizes, counts, delay_ms, opt):
    m = _network(sizes, counts, delay_ms, 17 + max(counts))
    with Simulation(m, log_synapse_events=1 << 20, **opt) as sim:
        tr, ev, syn, v = sim.run_all(), sim.read_events(), sim.read_synapse_events(), sim.voltages()
    (ref, ec, er, rv), (step, inst) = oracle.run_with_synapse_log(m)
    assert len(er) > 0 and len(step) > 0
    assert np.array_equal(tr, ref) and np.array_equal(v, rv)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
    assert np.array_equal(syn[0], step) and np.array_equal(syn[1], inst)
