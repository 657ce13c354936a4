"""Traces on both sides of the size up to which they are transposed on the host (256 KiB): equal rows,
with columns recorded out of order, twice, and many times over, in one chunk and in chunks."""
import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cells,rows,again", [(1, 1, 0), (64, 1023, 1), (64, 1024, 0), (64, 1025, 0), (3, 200, 400), (1000, 66, 3)])
@pytest.mark.parametrize("chunk", [0, 1, 65])
def test_rows_equal_the_oracle(cells, rows, again, chunk):
    m = configs.hh_population(n_cells=cells, t_final_ms=(rows - 1) * 0.025)
    m.record_comp = np.concatenate([np.arange(cells)[::-1], np.arange(again) % cells]).astype(np.int64)
    ref = oracle.run(m)[0]
    with Simulation(m, chunk_steps=chunk) as sim:
        assert np.array_equal(sim.run_all(), ref)
        tail, row0 = sim.read_trace()
        assert np.array_equal(tail, ref[row0:])
