"""Gate updates over the whole voltage range on the GPU, bit for bit against the oracle: inside
the range whose divisions run through double, outside it, at its edges, at rate midpoints and
next to them (where EXPLINEAR's 1 - exp(-x) vanishes), for every rate form, and for rates too
large or small for that range. The cells have a huge capacitance and no current, so each keeps
the voltage it starts from while its gates move."""
import numpy as np
import pytest

from eden_amd import _native as N
from eden_amd import configs
from eden_amd.model import Simulation, channel_type, rate
from oracle import oracle

pytestmark = pytest.mark.gpu

FORMS = {
    "squid": [(3, rate(N.RATE_EXPLINEAR, 1.0, -40.0, 10.0), rate(N.RATE_EXP, 4.0, -65.0, -18.0)),
              (1, rate(N.RATE_EXP, 0.07, -65.0, -20.0), rate(N.RATE_SIGMOID, 1.0, -35.0, 10.0))],
    "mid0": [(2, rate(N.RATE_EXPLINEAR, 0.5, 0.0, -4.0), rate(N.RATE_SIGMOID, 2.0, 0.0, -3.0)),
             (1, rate(N.RATE_FIXED, 0.3, 0.0, 1.0), rate(N.RATE_EXPLINEAR, 0.2, 1.5, 2.5), 3.0)],
    "extreme": [(1, rate(N.RATE_EXP, 1e7, -50.0, 5.0), rate(N.RATE_EXP, 1e-9, -50.0, -5.0)),
                (1, rate(N.RATE_SIGMOID, 0.0, -50.0, 5.0), rate(N.RATE_EXP, 0.1, -50.0, 1e-3))],
}


@pytest.mark.parametrize("name", sorted(FORMS))
def test_gates_at_every_voltage(name):
    gates = FORMS[name]
    f = np.float32
    edges = []
    for g in gates:
        for r in g[1:3]:
            for k in (0.0, 23.9, -23.9, 24.1, -24.1, 90.0, -90.0):
                c = f(r.midpoint) + f(k) * f(abs(r.scale))
                edges += [c, np.nextafter(c, f(np.inf)), np.nextafter(c, f(-np.inf))]
    v = np.concatenate([np.array(edges, f), np.linspace(-400, 400, 801).astype(f),
                        np.array([1e-3, -1e-3, 1e-7, -1e-7, 1e-20, 1e-39, -0.0], f)])
    m = configs.hh_population(n_cells=len(v), t_final_ms=1.0, amp_max_nA=0.0)
    m.channel_types = [channel_type([]), channel_type(gates), channel_type([])]
    n = len(v)
    m.v0 = v
    m.capacitance = np.full(n, 1e30, f)
    m.chan_gbase = np.zeros(3 * n, f)
    m.record_comp = np.repeat(np.arange(n), 1 + len(gates)).astype(np.int64)
    m.record_gate = np.tile(np.arange(-1, len(gates)), n).astype(np.int32)
    with Simulation(m) as sim:
        tr = sim.run_all()
    ref = oracle.run(m)[0]
    print(f"[gates] {name}: {n} voltages, {tr.shape[0]} rows", flush=True)
    assert np.array_equal(tr, ref, equal_nan=True)
