"""Launches with several lanes per electron (mcd_window.hip) against one lane
per electron: the same formulas step by step, so records, scatter rows and
counters are equal bit for bit.  The inline kernel (guard="inline", an explicit
block) begins with one lane per electron and gives several to the last 16 of a
wavefront; test_gpu_window_reference.py compares with kernels that do not."""
import numpy as np
import pytest

from mcd import _abi, engine

pytestmark = pytest.mark.gpu

COUNTED = [_abi.CNT_EVENTS, _abi.CNT_ELECTRONS, _abi.CNT_BKS, _abi.CNT_ABS, _abi.CNT_TRSM, _abi.CNT_LONG,
           _abi.CNT_FP64_PICKS, _abi.CNT_SCAT_ROWS, _abi.CNT_GUARD_TIMEOUTS]
INF = float("inf")


def _transport(material="Cu", E0=20000.0, Emin=1000.0, Wc=50.0, tilt=70.0, **kw):
    return engine.Transport(material, E0, Emin, Wc=Wc, s_tilt=tilt, tol_E=1e-2, tol_W=1e-2, grid_search="library", **kw)


# one lane per electron: FP64 to the end, continuous mode but for the last 16 of a wavefront
ONE_LANE = dict(block=256)
FP64 = _abi.PREC_FP64


def _same(a, b):
    assert a.els.tobytes() == b.els.tobytes()
    assert np.array_equal(a.counters[COUNTED], b.counters[COUNTED])
    if b.scats is not None:
        assert a.scats.tobytes() == b.scats.tobytes()


@pytest.fixture(scope="module")
def cu():
    return _transport()


# counts around which the lanes per electron change (256 CUs: 3840 << 6 = 7680 << 5
# = ..; one lane from 81921 on), one electron, one short of and past a wavefront
@pytest.mark.parametrize("n", [1, 3, 63, 65, 3840, 3841, 7680, 7681, 15361, 30720, 30721, 98304, 98305])
def test_ds_sizes_equal_one_lane_per_electron(cu, n):
    _same(cu.run(n, seed=n), cu.run(n, seed=n, guard="inline"))


@pytest.mark.parametrize("kw", [
    dict(material="Al", E0=5000.0, Emin=500.0, tilt=0.0),
    dict(material="Si", E0=1600.0, Wc=10.0, tilt=85.0),
    dict(material="Au", E0=30000.0, Wc=20.0, elastic="Ruth_nigram"),
    dict(material="Au", E0=5000.0, Emin=500.0, tilt=0.0, thickness=2000.0),
    dict(max_scatt=1), dict(max_scatt=63), dict(max_scatt=64), dict(max_scatt=65, thickness=20000.0, tilt=0.0),
], ids=str)
@pytest.mark.parametrize("n,first", [(5, (1 << 32) - 3), (700, 0), (20001, 17)])
def test_ds_configurations_equal_one_lane_per_electron(kw, n, first):
    tr = _transport(**kw)
    _same(tr.run(n, seed=4, first=first), tr.run(n, seed=4, first=first, guard="inline"))


@pytest.mark.parametrize("n,kept", [(1, 1), (70, 70), (300, 33)])
@pytest.mark.parametrize("kw", [dict(), dict(max_scatt=65), dict(material="Si", E0=10000.0, tilt=0.0, thickness=3000.0)],
                         ids=str)
def test_ds_scatter_rows_equal_one_lane_per_electron(kw, n, kept):
    tr = _transport(**kw)
    a = tr.run(n, seed=9, first=5, scats=True, scat_max_electron=5 + kept)
    _same(a, tr.run(n, seed=9, first=5, scats=True, scat_max_electron=5 + kept, guard="inline"))


def test_repeated_runs_are_equal(cu):
    a = cu.run(12345, seed=8)
    for _ in range(3):
        _same(cu.run(12345, seed=8), a)


# FP64 (DS): 1.5 wavefronts per SIMD to 8 lanes (98304 lanes), 4 to 4 lanes
@pytest.mark.parametrize("n", [1, 65, 1536, 1537, 12289, 65537])
def test_fp64_sizes_equal_one_lane_per_electron(cu, n):
    _same(cu.run(n, seed=n, precision=FP64), cu.run(n, seed=n, precision=FP64, **ONE_LANE))


@pytest.mark.parametrize("kw", [
    dict(material="Al", E0=5000.0, Emin=500.0, tilt=0.0, thickness=2000.0),
    dict(material="Au", E0=5000.0, Wc=20.0, elastic="Ruth_nigram"),
    dict(max_scatt=64), dict(max_scatt=1),
], ids=str)
def test_fp64_configurations_and_rows_equal_one_lane_per_electron(kw):
    tr = _transport(**kw)
    kw = dict(seed=3, first=(1 << 32) - 7, precision=FP64)
    _same(tr.run(1200, **kw), tr.run(1200, **kw, **ONE_LANE))
    kw.update(scats=True)
    _same(tr.run(40, **kw), tr.run(40, **kw, **ONE_LANE))


# continuous mode: one wavefront per SIMD (65536 lanes), quads to three (explicit law: to one)
@pytest.mark.parametrize("law", ["classical", "JL", "explicit"])
@pytest.mark.parametrize("n", [1, 65, 1024, 1025, 8193, 16384, 16385, 32769])
def test_continuous_sizes_equal_one_lane_per_electron(law, n):
    tr = engine.Transport("Au", 10000.0, 1000.0, s_tilt=70.0, mode="cont", bethe_model=law)
    _same(tr.run(n, seed=n), tr.run(n, seed=n, **ONE_LANE))


@pytest.mark.parametrize("kw", [
    dict(material="Cu", bethe_model="classical", thickness=20000.0, s_tilt=0.0),
    dict(material="Al", bethe_model="JL", elastic="Ruth_nigram", max_scatt=17),
    dict(material="Au", bethe_model="explicit", max_scatt=1),
    dict(material="Si", bethe_model="JL", thickness=800.0, max_scatt=64),
], ids=str)
def test_continuous_configurations_and_rows_equal_one_lane_per_electron(kw):
    tr = engine.Transport(kw.pop("material"), 10000.0, 1000.0, mode="cont", **{"s_tilt": 60.0, **kw})
    for n in (33, 9000):
        _same(tr.run(n, seed=3, first=9), tr.run(n, seed=3, first=9, **ONE_LANE))
    _same(tr.run(70, seed=3, scats=True, scat_max_electron=50), tr.run(70, seed=3, scats=True, scat_max_electron=50,
                                                                      **ONE_LANE))


# The last electrons of a large launch go on with several lanes each.  Forms
# without that: wavefront budgets other than 4 per SIMD.
@pytest.mark.parametrize("kw", [
    dict(),
    dict(material="Au", E0=30000.0, Wc=20.0),
    dict(material="Al", E0=5000.0, Emin=500.0, tilt=0.0, thickness=2000.0),
    dict(max_scatt=65), dict(max_scatt=1),
], ids=str)
@pytest.mark.parametrize("n,first", [(81921, 0), (131073, (1 << 32) - 60000), (400000, 9)])
def test_ds_drain_equals_one_lane_per_electron(kw, n, first):
    tr = _transport(**kw)
    a = tr.run(n, seed=4, first=first)
    _same(a, tr.run(n, seed=4, first=first, waves_per_simd=5))
    _same(tr.run(n, seed=4, first=first, block=64), a)


@pytest.mark.parametrize("n", [1, 16, 17, 700, 70000])
def test_drain_of_small_inline_launches(cu, n):
    _same(cu.run(n, seed=n, guard="inline"), cu.run(n, seed=n, guard="service"))
    tr = _transport(material="Si", E0=10000.0, thickness=9000.0, tilt=0.0)
    _same(tr.run(n, seed=n, guard="inline"), tr.run(n, seed=n, waves_per_simd=8))


@pytest.mark.parametrize("kw", [
    dict(material="Au", bethe_model="JL"), dict(material="Cu", bethe_model="classical", thickness=20000.0, s_tilt=0.0),
    dict(material="Au", bethe_model="explicit"), dict(material="Al", bethe_model="JL", max_scatt=17),
], ids=str)
@pytest.mark.parametrize("n", [17, 32769, 200000])
def test_continuous_drain_equals_one_lane_per_electron(kw, n):
    kw = dict(kw)
    tr = engine.Transport(kw.pop("material"), 10000.0, 1000.0, mode="cont", **{"s_tilt": 60.0, **kw})
    _same(tr.run(n, seed=3, first=9, block=256), tr.run(n, seed=3, first=9, waves_per_simd=5))


# the served guard: the last electrons' windows lie in the mailboxes, their guard picks are served
@pytest.mark.parametrize("kw", [
    dict(),
    dict(material="Au", E0=30000.0, Wc=20.0),
    dict(material="Al", E0=5000.0, Emin=500.0, tilt=0.0, thickness=2000.0),
    dict(max_scatt=65), dict(max_scatt=1),
], ids=str)
@pytest.mark.parametrize("n,first,shape", [(1, 0, {}), (961, 5, dict(block=128)), (40000, (1 << 32) - 60, dict(waves_per_simd=6)),
                                           (600001, 0, {})])
def test_ds_served_drain_equals_one_lane_per_electron(kw, n, first, shape):
    tr = _transport(**kw)
    _same(tr.run(n, seed=6, first=first, guard="service", **shape), tr.run(n, seed=6, first=first, waves_per_simd=5))


# the form with issue priorities begins at three wavefronts per SIMD (196608 electrons on 256 CUs)
@pytest.mark.parametrize("law", ["JL", "explicit"])
@pytest.mark.parametrize("n", [196607, 196608, 262145])
def test_continuous_priority_form_equals_the_others(law, n):
    tr = engine.Transport("Au", 6000.0, 1000.0, s_tilt=60.0, mode="cont", bethe_model=law)
    _same(tr.run(n, seed=3, first=9), tr.run(n, seed=3, first=9, waves_per_simd=5))


# quads to 3 wavefronts per SIMD (49152 electrons on 256 CUs), a kernel per screening on either side
@pytest.mark.parametrize("elastic", ["Ruth_vanilla", "Ruth_nigram"])
@pytest.mark.parametrize("law,n", [("JL", 49152), ("classical", 49153), ("JL", 196608), ("explicit", 16385)])
def test_continuous_screenings_equal_the_general_form(elastic, law, n):
    tr = engine.Transport("Au", 6000.0, 1000.0, s_tilt=60.0, mode="cont", bethe_model=law, elastic=elastic)
    _same(tr.run(n, seed=5, first=2), tr.run(n, seed=5, first=2, waves_per_simd=5))


# kernels with and without the tests for scatter rows, past the sizes of several lanes per electron
@pytest.mark.parametrize("kw,n", [(dict(), 81921), (dict(material="Au", E0=5000.0), 81921),
                                  (dict(material="Al", E0=5000.0, max_scatt=40), 90000)], ids=str)
def test_rows_do_not_change_the_records(kw, n):
    tr = _transport(**kw)
    for guard in ("inline", "service"):
        a = tr.run(n, seed=2, guard=guard)
        b = tr.run(n, seed=2, guard=guard, scats=True, scat_max_electron=50)
        assert a.els.tobytes() == b.els.tobytes()
        assert len(b.scats) == a.els["n_scatt"][:50].sum()
