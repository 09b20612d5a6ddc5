"""Several lanes per electron against kernels in which every electron keeps its
one lane to the end: FP32 at 5 wavefronts per SIMD, which have no windows for
their last electrons either (the inline kernel of the default budget has).  The
sizes are where the lanes per electron change on 256 CUs: DS 64 lanes up to
3.75 x 65536 lanes in all, .. 8 up to 30720 electrons, 4 up to 81920; continuous
mode 64 lanes up to 65536 lanes, .. 8 up to 8192 electrons, 4 up to 49152
(explicit law 16384)."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import _abi, engine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]

COUNTED = [_abi.CNT_EVENTS, _abi.CNT_ELECTRONS, _abi.CNT_BKS, _abi.CNT_ABS, _abi.CNT_TRSM, _abi.CNT_LONG,
           _abi.CNT_FP64_PICKS]


def _ds(material="Cu", E0=20000.0, Emin=1000.0, Wc=50.0, tilt=70.0, **kw):
    return engine.Transport(material, E0, Emin, Wc=Wc, s_tilt=tilt, tol_E=1e-2, tol_W=1e-2, grid_search="library", **kw)


def _equal(tr, n, first=0, **kw):
    a, b = tr.run(n, seed=n, first=first, **kw), tr.run(n, seed=n, first=first, waves_per_simd=5)
    same = a.els.tobytes() == b.els.tobytes()
    assert same and np.array_equal(a.counters[COUNTED], b.counters[COUNTED])


@pytest.mark.parametrize("n", [1, 3, 63, 65, 3840, 3841, 7680, 7681, 15360, 15361, 30720, 30721, 81920, 81921])
def test_ds_sizes(n):
    tr = _ds(E0=8000.0)
    _equal(tr, n)
    _equal(tr, n, guard="inline")
    _equal(tr, n, guard="service")


@pytest.mark.parametrize("kw", [
    dict(material="Al", E0=5000.0, Emin=500.0, tilt=0.0),
    dict(material="Si", E0=1600.0, Wc=10.0, tilt=85.0),
    dict(material="Au", E0=30000.0, Wc=20.0, elastic="Ruth_nigram"),
    dict(material="Au", E0=5000.0, Emin=500.0, tilt=0.0, thickness=2000.0),
    dict(max_scatt=1), dict(max_scatt=63), dict(max_scatt=64), dict(max_scatt=65, thickness=20000.0, tilt=0.0),
], ids=str)
@pytest.mark.parametrize("n,first", [(5, (1 << 32) - 3), (700, 0), (20001, 17), (81920, 3)])
def test_ds_configurations(kw, n, first):
    _equal(_ds(**kw), n, first)


@pytest.mark.parametrize("law,most", [("classical", 49152), ("JL", 49152), ("explicit", 16384)])
@pytest.mark.parametrize("n", [1, 65, 1024, 1025, 2049, 4097, 8192, 8193, 0, -1])
def test_continuous_sizes(law, most, n):
    tr = engine.Transport("Au", 10000.0, 1000.0, s_tilt=70.0, mode="cont", bethe_model=law)
    n = n if n > 0 else most - n
    _equal(tr, n)
    _equal(tr, n, block=256)


@pytest.mark.parametrize("kw", [
    dict(material="Cu", bethe_model="classical", thickness=20000.0, s_tilt=0.0),
    dict(material="Al", bethe_model="JL", elastic="Ruth_nigram", max_scatt=17),
    dict(material="Au", bethe_model="explicit", max_scatt=1),
    dict(material="Si", bethe_model="JL", thickness=800.0, max_scatt=64),
], ids=str)
@pytest.mark.parametrize("n", [33, 9000, 16384])
def test_continuous_configurations(kw, n):
    kw = dict(kw)
    _equal(engine.Transport(kw.pop("material"), 10000.0, 1000.0, mode="cont", **{"s_tilt": 60.0, **kw}), n, 9)
