"""kernel_infos names the kernel that runs a bucket, as a profiler lists it: the lean kernel for
passive trees on active somata, the general one where a dendrite is recorded (whose constant-tree
form, with and without a channel wave and in every workgroup size, equals the oracle here), its
forms for long synapse lists and for cells whose gate table is not in LDS, and the point kernels."""
import dataclasses

import numpy as np
import pytest

from eden_amd import configs
from eden_amd.model import Simulation
from oracle import oracle

pytestmark = pytest.mark.gpu


def _symbols(m, **opt):
    with Simulation(m, **opt) as sim:
        tr = sim.run_all()
        infos = sim.kernel_infos()
    assert np.array_equal(tr, oracle.run(m)[0])
    assert all(k["name"].split("<")[0] in k["symbol"] for k in infos)
    return sorted(k["symbol"] for k in infos)


@pytest.mark.parametrize("threads", [64, 128, 256, 512])
@pytest.mark.parametrize("wave", [1, -1])
@pytest.mark.parametrize("recorded", [False, True])
def test_passive_trees(threads, wave, recorded):
    m = configs.random_trees(sizes=[20, 130, 250], n_cells=3, t_final_ms=12.0, seed=threads)
    if recorded:
        m = dataclasses.replace(m, record_comp=np.concatenate([m.record_comp, m.cell_comp_begin[1:] - 1]))
    split = "true" if wave > 0 else "false"
    want = f"tree_kernel<{threads}, {split}, false>" if recorded else f"lean_tree_kernel<{threads}, {split}>"
    assert _symbols(m, threads_per_cell=threads, channel_wave=(wave,) * 4) == [want]


def test_other_kernels():
    trees = configs.random_trees(sizes=[60, 300], n_cells=2, t_final_ms=3.0, seed=5, hh_everywhere=True)
    assert _symbols(trees) == ["tree_kernel<128, false, false>", "tree_kernel<64, true, false>"]
    large = configs.random_trees(sizes=[1880], n_cells=1, t_final_ms=1.0, seed=5, hh_everywhere=True)
    large = dataclasses.replace(large, channel_types=list(large.channel_types) + [large.channel_types[1]] * 61)
    assert _symbols(large) == ["tree_kernel<513, true, false>"]
    assert _symbols(configs.hh_population(n_cells=9, t_final_ms=2.0)) == ["point_quad_kernel"]
    net = configs.mixed_network(tree_sizes=(30, 90), n_point=3, n_conn=30, t_final_ms=3.0)
    assert _symbols(net) == ["point_kernel", "tree_kernel<128, false, true>", "tree_kernel<64, false, true>"]
    # the same instances, all on the first tree's soma
    at = np.zeros(net.n_comps + 1, np.int64)
    at[1:] = net.n_synapses
    long = dataclasses.replace(net, comp_syn_begin=at, syn_type=np.sort(net.syn_type))
    assert net.n_synapses >= 16
    assert _symbols(long) == ["point_kernel", "tree_kernel<128, false, true>", "tree_kernel<66, false, true>"]
    assert _symbols(long, network_window=-1) == ["point_kernel", "tree_kernel<70, false, true>"]
    cells = configs.spiking_network(n_cells=40, in_degree=17, t_final_ms=3.0)
    assert _symbols(cells)[0] in ("net_quad_kernel<2>", "net_quad_kernel<4>")
