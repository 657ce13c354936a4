"""Cells near the limit of a workgroup's LDS: HH channels on every compartment in models of 3 to 64
channel types, at sizes where the gate table does not fit beside the cell's other tables and is
read from global memory, with and without a channel wave and in a network. Every cell is accepted
and its traces and last voltages equal the oracle's."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu
CU_LDS = 160 * 1024


def _with_types(m, types):
    """The model with its channel types up to `types`, the HH ones repeated, and its
    compartments' channels spread over the repetitions."""
    base = list(m.channel_types)
    kind = np.asarray(m.chan_type)
    again = 1 + np.arange(types - len(base)) % 2          # of channel types 1 and 2
    copies = {k: np.concatenate([[k], len(base) + np.flatnonzero(again == k)]) for k in (1, 2)}
    moved = kind.copy()
    for k in (1, 2):
        at = np.flatnonzero(kind == k)
        moved[at] = copies[k][np.arange(len(at)) % len(copies[k])]
    return dataclasses.replace(m, channel_types=base + [base[k] for k in again], chan_type=moved)


def _parents(shape, n):
    rng = np.random.default_rng(11)
    if shape == "chain":
        return np.arange(-1, n - 1, dtype=np.int32)
    if shape == "binary":
        return np.array([-1] + [(i - 1) // 2 for i in range(1, n)], np.int32)
    return np.array([-1] + [int(rng.integers(max(0, i - 40), i)) for i in range(1, n)], np.int32)


def _check(m, types, **opt):
    with Simulation(m, **opt) as sim:
        tr, ev, v = sim.run_all(), sim.read_events(), sim.voltages()
        lds = max(k["lds_bytes"] for k in sim.kernel_infos())
    # 64 bytes a table entry, four entries a type
    assert lds <= CU_LDS < lds + 64 * 4 * types + 64
    ref, ec, er, rv = oracle.run(m)
    assert np.array_equal(tr, ref), float(np.abs(tr - ref).max())
    assert np.array_equal(v, rv)
    assert np.array_equal(ev[0], ec) and np.array_equal(ev[1], er)


@pytest.mark.parametrize("shape,types,n,wave", [
    ("random", 3, 1882, 0), ("random", 16, 1863, 0), ("random", 64, 1791, 0), ("random", 64, 1700, -1), ("chain", 64, 1649, 0),
    ("binary", 64, 1840, 0), ("binary", 16, 1913, 0)])
def test_cells_whose_gate_table_is_in_global_memory(shape, types, n, wave):
    m = configs.random_trees(parents=[_parents(shape, n)], t_final_ms=1.0, seed=9, hh_everywhere=True)
    m = dataclasses.replace(m, pulse_start=np.full(1, 100.0, np.float32), record_comp=np.arange(0, n, 7))
    _check(_with_types(m, types), types, channel_wave=(wave,) * 4)


def test_network_cell_whose_gate_table_is_in_global_memory():
    m = configs.mixed_network(tree_sizes=(1840, 1800, 60), n_point=3, n_conn=40, t_final_ms=4.0, seed=4, hh_everywhere=True,
                              delay_ms=(0.5, 1.0), weight=(3.0, 9.0))
    m = dataclasses.replace(m, pulse_start=np.full(len(m.pulse_start), 100.0, np.float32))
    _check(_with_types(m, 64), 64)
