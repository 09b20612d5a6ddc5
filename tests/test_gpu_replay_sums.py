"""How well the derivative replay repeats: its sums over electrons are FP32 in a
lane and over a wavefront's lanes, FP64 over wavefronts."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import _abi, engine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]

# One electron per lane (by position): only the order of the wavefronts in the
# FP64 sum varies.  The order of a sum of N terms (at most 256 CUs x 24
# wavefronts) moves it by less than 2 N 2^-53 times the sum of the magnitudes.
TOL_ONE = 2 * 6144 * 2.0 ** -53
# More electrons than lanes: which electrons a lane adds up varies.  An addition
# to a lane sum of a few electrons' magnitude (4 here) is rounded by 2^-24 of it
# at most, with either sign: the lanes' 2000 additions each add up as a random
# walk; 6 standard deviations of the difference of two runs.
LANES = 256 * 24 * 64


def tol_many(n):
    return 6 * np.sqrt(2 * LANES * 2000) * 2.0 ** -24 * 4 / n


@pytest.mark.parametrize("n", [1, 65, 100001, 1 << 19])
@pytest.mark.parametrize("kw", [dict(Wc=50.0, tol_E=1e-2, tol_W=1e-2), dict(mode="cont", bethe_model="JL")],
                         ids=["ds", "cont"])
def test_repeated_products_are_equal_to_rounding(kw, n):
    import torch
    tr = engine.Transport("Cu", 6000.0, 1000.0, s_tilt=70.0, **kw)
    g = torch.from_numpy(np.random.default_rng(1).standard_normal(65).astype(np.float32)).cuda()

    def sums(n, first=0):
        out = torch.zeros(1 + _abi.NGRAD, dtype=torch.float64, device="cuda")
        tr.vjp(n, g, out=out, seed=3, first=first)
        return out.cpu().numpy()

    # the terms' magnitudes, from single electrons
    size = n * np.mean([np.abs(sums(1, first=e)) for e in range(400)], axis=0)
    tol = (TOL_ONE if n < 200000 else tol_many(n)) * size
    a = sums(n)
    assert np.isfinite(a).all()
    for _ in range(6):
        b = sums(n)
        assert (np.abs(b - a) <= tol).all(), (b - a) / np.maximum(size, 1e-300)


# The replay's forms on 256 CUs: issue priorities from 131072 electrons (not for
# Si 5 keV), one electron per lane up to 327680 (DS) and 393216, none of both in
# continuous mode from 16 electrons per lane.  Float32 sums of up to ~10^4 terms
# per lane and bin: within 1e-4 of the sum of magnitudes.
@pytest.mark.parametrize("n", [131071, 131072, 327680, 327681, 393216, 393217, 16 * 393216])
@pytest.mark.parametrize("kw", [dict(material="Cu", Wc=50.0, tol_E=1e-2, tol_W=1e-2),
                                dict(material="Au", mode="cont", bethe_model="JL"),
                                dict(material="Si", mode="cont", bethe_model="classical")], ids=str)
def test_products_equal_jacobians_in_every_form(kw, n):
    import torch
    if kw["material"] == "Cu" and n > 400000:
        n = 400000
    kw = dict(kw)
    tr = engine.Transport(kw.pop("material"), 5000.0, 1000.0, s_tilt=60.0, **kw)
    g = np.random.default_rng(2).standard_normal(65).astype(np.float32)
    J, out = np.asarray(tr.jacobian(n, seed=5)), np.asarray(tr.vjp(n, torch.from_numpy(g), seed=5))
    assert J[0, 0] > 0 and np.isfinite(J).all()
    want, size = g.astype(np.float64) @ J, np.abs(g).astype(np.float64) @ np.abs(J)
    assert (np.abs(out - want) <= 1e-4 * np.maximum(size, np.abs(J).sum() * 1e-3)).all()
    # the same electrons in two launches
    h = n // 2
    halves = (np.asarray(tr.jacobian(h, seed=5)) * h + np.asarray(tr.jacobian(n - h, seed=5, first=h)) * (n - h)) / n
    assert (np.abs(halves - J) <= 1e-4 * np.maximum(np.abs(J), np.abs(J).sum() * 1e-3)).all()
