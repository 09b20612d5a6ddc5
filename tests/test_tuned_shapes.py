"""Which launches use a tuned shape, and what the tuners choose from."""
import ctypes as C
from types import SimpleNamespace

import pytest

from conftest import gpu_available
from mcd import _abi, autotune, engine

SHAPE = dict(block=1024, waves_per_simd=8, guard="service", refill_period=2)


def _launched(monkeypatch, mode, law, tuned, n, **kw):
    """(block, waves_per_simd, flags) that a launch hands to the library."""
    got = {}

    def forward(ctx, cfg, tables, seed, config_id, first, n, els, scats, counters, launch, stream):
        la = C.cast(launch, C.POINTER(_abi.Launch)).contents
        got.update(block=la.block, waves=la.waves_per_simd, flags=la.flags)
        return 0

    monkeypatch.setattr(engine, "lib", lambda: SimpleNamespace(mcd_forward=forward))
    monkeypatch.setattr(engine, "context", lambda device=0: None)
    monkeypatch.setattr(engine.torch.cuda, "get_device_properties",
                        lambda device: SimpleNamespace(multi_processor_count=256))
    tr = object.__new__(engine.Transport)
    tr.device, tr.mode, tr.tuned, tr._tables = 0, mode, tuned, None
    tr.cfg = _abi.Config()
    tr.cfg.mode, tr.cfg.bethe_model = mode, law
    buf = SimpleNamespace(data_ptr=lambda: 0)
    tr.launch(n, buf, buf, stream=SimpleNamespace(cuda_stream=0), **kw)
    return got["block"], got["waves"], got["flags"]


# the largest launches with several lanes per electron on 256 CUs
@pytest.mark.parametrize("mode,law,small", [(_abi.MODE_DS, _abi.BETHE_CLASSICAL, 81920),
                                            (_abi.MODE_CONT, _abi.BETHE_JL, 49152),
                                            (_abi.MODE_CONT, _abi.BETHE_EXPLICIT, 16384)])
def test_a_shape_of_large_launches_is_not_used_for_small_ones(monkeypatch, mode, law, small):
    flags = engine.guard_flags("service") | engine.refill_flags(2)
    large = dict(SHAPE, n=1 << 22)
    assert _launched(monkeypatch, mode, law, large, small) == (0, 0, 0)
    assert _launched(monkeypatch, mode, law, large, small + 1) == (1024, 8, flags)
    # tuned at a small size, or set by hand: used throughout
    assert _launched(monkeypatch, mode, law, dict(SHAPE, n=small), small) == (1024, 8, flags)
    assert _launched(monkeypatch, mode, law, dict(SHAPE, n=small), 1 << 22) == (1024, 8, flags)
    assert _launched(monkeypatch, mode, law, SHAPE, 7) == (1024, 8, flags)
    # what the caller names stays
    assert _launched(monkeypatch, mode, law, large, small, block=128) == (128, 0, 0)


def test_the_tuners_try_the_librarys_own_shape():
    assert dict(block=0, waves_per_simd=0, guard=None, refill_period=1) in autotune.TRANSPORT_CANDIDATES
    for nodes in (0, 128):
        assert any(c["block"] == 0 and c["pick_nodes"] == nodes for c in autotune.CANDIDATES)


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="no GPU")
@pytest.mark.parametrize("kw", [dict(Wc=50.0, tol_E=1e-2, tol_W=1e-2), dict(mode="cont", bethe_model="JL")],
                         ids=["ds", "cont"])
def test_tuning_a_small_launch_can_keep_several_lanes_per_electron(kw):
    tr = engine.Transport("Cu", 20000.0, 1000.0, s_tilt=70.0, **kw)
    ref = tr.run(10007, seed=2)
    res = tr.tune(10007, use_cache=False)
    # a step of one lane per electron takes over twice as long
    assert (tr.tuned["block"], tr.tuned["guard"], tr.tuned["n"]) == (0, None, 10007), res["ms"]
    assert tr.run(10007, seed=2).els.tobytes() == ref.els.tobytes()
    assert tr.run(100001, seed=2).els.tobytes() == tr.run(100001, seed=2, waves_per_simd=5).els.tobytes()


@pytest.mark.gpu
@pytest.mark.skipif(not gpu_available(), reason="no GPU")
def test_an_asked_for_register_budget_is_a_shape(monkeypatch):
    """MCD_MINW sets the wavefronts per SIMD of small launches too: one lane per
    electron, over three times as long for 10007 electrons."""
    import torch
    tr = engine.Transport("Cu", 20000.0, 1000.0, s_tilt=70.0, Wc=50.0, tol_E=1e-2, tol_W=1e-2)
    n = 10007
    els = torch.empty(n * _abi.ELECTRON_DTYPE.itemsize, dtype=torch.uint8, device="cuda")
    cnt = torch.zeros(_abi.NCOUNTERS, dtype=torch.int64, device="cuda")

    def best():
        t = []
        for _ in range(4):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            tr.launch(n, els, cnt)
            b.record()
            torch.cuda.synchronize()
            t.append(a.elapsed_time(b))
        return min(t), els.cpu().numpy().tobytes()

    own, rec = best()
    monkeypatch.setenv("MCD_MINW", "5")
    asked, same = best()
    equal = same == rec
    assert equal and asked > 2 * own, (asked, own)
