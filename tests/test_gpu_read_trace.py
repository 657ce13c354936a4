"""Traces read back in pieces through the device's transposition: row and column counts around
its 64 x 64 tiles, a column recorded twice, a single column, chunked runs, and rows that take
several pieces; equal to the oracle's. A rewound model gives the same results again, also
when it is read or saved right after the rewind."""
import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,rows,chunk", [(1, 1, 0), (63, 64, 0), (64, 65, 0), (65, 63, 17), (130, 201, 64)])
def test_rows_equal_the_oracle(cells, rows, chunk):
    m = configs.hh_population(n_cells=cells, t_final_ms=(rows - 1) * 0.025)
    m.record_comp = np.concatenate([np.arange(cells)[::-1], [0]]).astype(np.int64)
    ref = oracle.run(m)[0]
    with Simulation(m, chunk_steps=chunk) as sim:
        first = sim.get_state()
        tr = sim.run_all()
        v = sim.voltages()
        sim.reset()
        assert sim.get_state() == first
        assert np.array_equal(sim.voltages(), m.v0)
        again = sim.run_all()
    print(f"[read] {cells} cells, {rows} rows, chunk {chunk}", flush=True)
    assert tr.shape == (rows, cells + 1)
    assert np.array_equal(tr, ref) and np.array_equal(again, ref)
    assert np.array_equal(v, v) and v.shape == (cells,)


def test_trace_of_several_pieces():
    """2,000 rows of 3,000 columns (24 MB) pass the 16 MiB staging buffer twice."""
    m = configs.hh_population(n_cells=3000, t_final_ms=49.975)
    with Simulation(m) as sim:
        tr = sim.run_all()
        tail, row0 = sim.read_trace()
    assert row0 == 0 and np.array_equal(tr, tail)
    pick = np.array([0, 1, 1499, 2999])
    sub = m.subset(pick)[0]
    assert np.array_equal(tr[:, pick], oracle.run(sub)[0])
