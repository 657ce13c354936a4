"""The size-limit autotuner on a network of tree cells, with a fake timer: the search starts from
the limits that the library chose for the network and can keep or reach each of its candidates."""
import pytest

from eden_amd import autotune, configs

WINDOW, SINGLE = (64, 128, 512, 2047), (256, 512, 512, 2047)


def _tune(monkeypatch, rule, timing):
    m = configs.mixed_network(tree_sizes=(30, 100, 300), n_point=4, n_conn=20, t_final_ms=1.0)
    calls = []

    class Context:
        def __init__(self, model, device=0):
            assert model is m

        def __enter__(self):
            return self

        def __exit__(self, *a):
            pass

        def size_limits(self):
            return rule

    def fake(model, limits, steps=None, repeats=2, device=0):
        calls.append(tuple(limits))
        return timing(tuple(limits))

    monkeypatch.setattr(autotune, "Simulation", Context)
    monkeypatch.setattr(autotune, "time_limits", fake)
    limits, report = autotune.autotune(m)
    assert [l for l, _ in report] == calls
    return limits, calls


@pytest.mark.parametrize("rule", [WINDOW, SINGLE])
def test_network_keeps_the_librarys_limits(monkeypatch, rule):
    limits, calls = _tune(monkeypatch, rule, lambda l: 1.0)
    assert limits == rule and calls[0] == rule
    assert all(c[i] <= c[i + 1] for c in calls for i in range(3))


@pytest.mark.parametrize("rule", [WINDOW, SINGLE])
def test_network_search_never_ends_slower_than_it_started(monkeypatch, rule):
    # wider limits are slower, as for trees whose launches run several steps
    limits, calls = _tune(monkeypatch, rule, lambda l: float(sum(l[:3])))
    assert sum(limits) <= sum(rule)
    limits, calls = _tune(monkeypatch, rule, lambda l: 0.5 if l[1] == 256 else 1.0)
    assert limits[1] == 256
