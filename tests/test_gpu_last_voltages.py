"""Every cell's voltage after a run equals the oracle's, also of cells that are not recorded, where it
passes through more than one place: windowed networks (two copies of the state, an odd or even
number of windows in a chunk, chunks of one step, windows run again step by step), point cells read
by chunks, and trees; after a rewind and a second run too."""
import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle
from tests.test_gpu_net_quad import _network

pytestmark = pytest.mark.gpu


def _check(m, **opt):
    rv = oracle.run(m)[3]
    with Simulation(m, **opt) as sim:
        assert np.array_equal(sim.voltages(), m.v0)
        for again in (False, True):
            sim.run_all()
            assert np.array_equal(sim.voltages(), rv), again
            sim.reset()
        assert np.array_equal(sim.voltages(), m.v0)


@pytest.mark.parametrize("types,synapses", [(2, 30), (5, 30)])     # four lanes a cell, one lane a cell
@pytest.mark.parametrize("opt", [{}, dict(chunk_steps=39), dict(chunk_steps=1), dict(chunk_steps=77), dict(network_window=-2),
                                 dict(network_window=-1), dict(network_window=5, chunk_steps=13)])
def test_networks(types, synapses, opt):
    _check(_network(33, synapses // 2, synapses, types, 1, 7), **opt)


@pytest.mark.parametrize("chunk", [0, 1, 64])
def test_uncoupled_cells(chunk):
    _check(configs.hh_population(n_cells=130, t_final_ms=2.0), chunk_steps=chunk)
    _check(configs.random_trees(sizes=[1, 2, 70, 300, 1100], n_cells=5, t_final_ms=1.0, seed=4), chunk_steps=chunk)
    _check(configs.random_trees(sizes=[1, 2, 70, 300, 1100], n_cells=5, t_final_ms=1.0, seed=4, hh_everywhere=True),
           chunk_steps=chunk)
