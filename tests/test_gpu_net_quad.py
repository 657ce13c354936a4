"""The windowed network kernel with four lanes per cell, and the forms it leaves to one lane per
cell: traces, spike raster, every synaptic delivery and every cell's last voltage equal the
oracle's, over synapse counts around its groups of 16, several types in a cell, cells without
synapses of a type or without any, cell counts around its waves, and up to five Poisson
inputs a cell."""
import dataclasses

import numpy as np
import pytest

from eden_amd import _native as N
from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
MS = 1000.0


def _network(n, lo, hi, types, poisson, seed):
    """n HH cells, lo to hi synapses each over `types` types, `poisson` Poisson inputs each."""
    rng = np.random.default_rng(seed)
    m = configs.hh_population(n_cells=n, t_final_ms=20.0, seed=seed, amp_max_nA=0.3)
    m.pulse_start = np.full(n, 2.0 * MS, np.float32)
    cnt = rng.integers(lo, hi + 1, n)
    cnt[0], cnt[-1] = lo, hi
    begin = np.concatenate([[0], np.cumsum(cnt)]).astype(np.int64)
    ns = int(begin[-1])
    stype = np.concatenate([np.sort(rng.integers(0, types, c)) for c in cnt]).astype(np.int32)
    if n > 2:
        stype[begin[1]:begin[2]] = types - 1          # a cell with one type only
    pre = rng.integers(0, n, ns)
    order = np.argsort(pre, kind="stable")
    spikes = np.concatenate([[0], np.cumsum(np.bincount(pre, minlength=n))]).astype(np.int64)
    st = [N.ExpTwoType(1e-3 * (1 + t), (0.0, -80.0)[t % 2], 500.0 + 77.0 * t, 5000.0 + 333.0 * t, 1.0)
          for t in range(types)]
    k = n * poisson
    return dataclasses.replace(
        m, syn_types=st, comp_syn_begin=begin, syn_type=stype, syn_weight=rng.uniform(0.5, 3.0, ns).astype(np.float32),
        syn_delay=(np.round(rng.uniform(1.0, 4.0, ns) * MS / 25.0) * 25.0).astype(np.float32),
        comp_spike_begin=spikes, spike_target=order.astype(np.int64),
        comp_poisson_begin=np.arange(n + 1, dtype=np.int64) * poisson, poisson_rate=np.full(k, 3e-4, np.float32),
        poisson_syn_type=np.tile(np.arange(poisson, dtype=np.int32) % types, n),
        poisson_weight=rng.uniform(0.5, 2.0, k).astype(np.float32),
        poisson_instance=np.tile(np.arange(poisson, dtype=np.int32), n), poisson_rng_offset=np.zeros(k, np.int32))


@pytest.mark.parametrize("n,lo,hi,types,poisson,quad", [
    (1, 1, 1, 1, 0, True), (17, 0, 3, 2, 1, True), (33, 15, 17, 1, 2, True), (16, 30, 33, 2, 4, True),
    (70, 0, 120, 4, 3, True), (40, 60, 130, 3, 1, True), (20, 180, 200, 2, 0, False), (20, 180, 200, 1, 0, True), (65, 200, 256, 4, 1, False),
    (30, 10, 40, 2, 5, False), (1, 256, 256, 1, 1, True)])
def test_network_kernels_bit_exact(n, lo, hi, types, poisson, quad):
    m = _network(n, lo, hi, types, poisson, seed=100 + n)
    with Simulation(m, log_synapse_events=1 << 20, chunk_steps=301, profile=True) as sim:
        tr = sim.run_all()
        ev = sim.read_events()
        step, syn = sim.read_synapse_events()
        v = sim.voltages()
        deliveries = sim.network_stats()[3]
        name = sim.kernel_infos()[0]["name"]
    (rt, ec, er, rv), (ostep, osyn) = oracle.run_with_synapse_log(m)
    print(f"[net] n={n} synapses {lo}-{hi} types {types} poisson {poisson}: {name}, {len(er)} spikes, "
          f"{len(ostep)} deliveries", flush=True)
    assert name == ("net_quad_kernel" if quad else "net_window_kernel")
    assert np.array_equal(tr, rt)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)
    assert np.array_equal(step, ostep) and np.array_equal(syn, osyn) and deliveries == len(ostep)
