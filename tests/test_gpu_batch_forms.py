"""The batched kernel's inline forms: with a drain (runs that end in their
longest trajectories) and without (workgroups of one wavefront where LDS holds
more of them), against per-configuration launches bit for bit."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import _abi, engine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]


def _check(items, nodes, **kw):
    b = engine.Batch(items, pick_nodes=nodes)
    for use_graph in (False, True):
        b.counters.zero_()
        b.launch(seed=3, use_graph=use_graph, **kw)
        for i, ((tr, n), r) in enumerate(zip(items, b.results())):
            if n == 0:
                continue
            ref = tr.run(n, seed=3, config_id=i, waves_per_simd=5)
            assert r.els.tobytes() == ref.els.tobytes(), i
            assert int(r.counters[_abi.CNT_EVENTS]) == ref.events
            assert int(r.counters[_abi.CNT_FP64_PICKS]) == int(ref.counters[_abi.CNT_FP64_PICKS])


def _items(ns, nodes):
    kw = dict(tol_E=1e-2, tol_W=1e-2, grid_search="library", pick_nodes=nodes)
    trs = [engine.Transport("Au", 8000.0, 1000.0, Wc=20.0, s_tilt=70.0, **kw),
           engine.Transport("Au", 10000.0, 1000.0, s_tilt=0.0, mode="cont", bethe_model="explicit"),
           engine.Transport("Al", 5000.0, 500.0, s_tilt=0.0, thickness=2000.0, **kw),
           engine.Transport("Si", 6000.0, 1000.0, s_tilt=60.0, mode="cont", bethe_model="JL"),
           engine.Transport("Cu", 5000.0, 1000.0, s_tilt=45.0, max_scatt=65, **kw)]
    return [(tr, n) for tr, n in zip(trs, ns)]


@pytest.mark.parametrize("ns", [(1, 0, 17, 16, 15), (64, 65, 3, 700, 1), (20001, 5000, 30000, 40000, 50000)])
@pytest.mark.parametrize("kw", [dict(), dict(block=64), dict(block=128), dict(refill_period=4)], ids=str)
@pytest.mark.parametrize("nodes", [128, 157])
def test_short_runs_equal_per_configuration_launches(ns, kw, nodes):
    _check(_items(ns, nodes), nodes, **kw)


# more than ten trajectories for each of the 16 x 64 lanes per CU
@pytest.mark.parametrize("kw", [dict(), dict(block=256), dict(block=128)], ids=str)
def test_long_runs_equal_per_configuration_launches(kw):
    common = dict(tol_E=1e-2, tol_W=1e-2, grid_search="library", pick_nodes=227)
    items = [(engine.Transport("Cu", 1400.0, 1000.0, s_tilt=30.0, **common), 1800000),
             (engine.Transport("Al", 1300.0, 1000.0, s_tilt=0.0, **common), 1900001),
             (engine.Transport("Si", 1500.0, 1000.0, s_tilt=60.0, mode="cont"), 5000)]
    _check(items, 227, **kw)
