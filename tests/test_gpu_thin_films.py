"""Films thinner than a free path of the grazing beam: every form with several
lanes per electron against the kernels that have one lane per electron to the
end (FP32: 5 wavefronts per SIMD; FP64: one kernel for an explicit block)."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import _abi, engine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]

COUNTED = [_abi.CNT_EVENTS, _abi.CNT_ELECTRONS, _abi.CNT_BKS, _abi.CNT_ABS, _abi.CNT_TRSM, _abi.CNT_LONG,
           _abi.CNT_FP64_PICKS]
DS = dict(Wc=20.0, tol_E=1e-2, tol_W=1e-2, grid_search="library")
MODES = {"ds": DS, "classical": dict(mode="cont", bethe_model="classical"), "JL": dict(mode="cont", bethe_model="JL"),
         "explicit": dict(mode="cont", bethe_model="explicit")}


def _film(thickness, mode="ds", **kw):
    return engine.Transport("Au", 5000.0, 1000.0, s_tilt=85.0, thickness=thickness, **MODES[mode], **kw)


def _same(a, b, thickness):
    # electrons inside after several steps: what a window of whole steps in the film needs
    assert len(b.els) < 1000 or (b.els["n_scatt"] > 5).any()
    z = b.els["pos"][:, 2]
    assert ((z >= 0) & (z < thickness)).all()
    equal = a.els.tobytes() == b.els.tobytes()
    assert equal
    assert np.array_equal(a.counters[COUNTED], b.counters[COUNTED])


# 64, 32, .. 4 lanes per electron, one lane per electron with the last ones' windows
@pytest.mark.parametrize("n", [40, 3001, 9000, 20001, 60000, 81920, 200001])
@pytest.mark.parametrize("thickness", [1.0, 0.5, 1.5])
def test_ds_films(n, thickness):
    tr = _film(thickness)
    b = tr.run(n, seed=n, waves_per_simd=5)
    _same(tr.run(n, seed=n), b, thickness)
    _same(tr.run(n, seed=n, guard="inline"), b, thickness)
    _same(tr.run(n, seed=n, guard="service"), b, thickness)


@pytest.mark.parametrize("n", [40, 2001, 12000, 16384, 200001])
@pytest.mark.parametrize("thickness", [1.0, 0.5])
@pytest.mark.parametrize("mode", ["classical", "JL", "explicit"])
def test_continuous_films(mode, thickness, n):
    tr = _film(thickness, mode)
    b = tr.run(n, seed=n, waves_per_simd=5)
    _same(tr.run(n, seed=n), b, thickness)
    _same(tr.run(n, seed=n, block=256), b, thickness)


@pytest.mark.parametrize("n", [40, 3001, 12000, 65536])
@pytest.mark.parametrize("thickness", [1.0, 0.5])
def test_fp64_films(thickness, n):
    tr = _film(thickness)
    kw = dict(seed=n, precision=_abi.PREC_FP64)
    _same(tr.run(n, **kw), tr.run(n, block=256, **kw), thickness)


def test_batched_films():
    items = [(_film(1.0, pick_nodes=128), 9000), (_film(0.5, pick_nodes=128), 30001), (_film(1.0, "JL"), 20000),
             (_film(0.5, "explicit"), 20000)]
    b = engine.Batch(items, pick_nodes=128)
    b.launch(seed=3)
    for i, ((tr, n), r) in enumerate(zip(items, b.results())):
        _same(r, tr.run(n, seed=3, config_id=i, waves_per_simd=5), tr.cfg.thickness)
