"""The derivative replay's kernels, one per channel count: the vector-Jacobian
product against the Jacobian of the same streams, and the values against the
sum over the histogram."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import engine
from mcd.material import Material

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]


# float32 sums of up to ~10^4 terms per bin: their error stays within 1e-4 of the sum of magnitudes
@pytest.mark.parametrize("n_bins", [1, 64, 256])
@pytest.mark.parametrize("shells", [1, 2, 3, 4, 5, 6, 7, 8, None])
def test_vjp_equals_jacobian_for_every_channel_count(shells, n_bins):
    import torch
    mat = Material("Au")
    kw = dict(mode="cont", bethe_model="JL")
    if shells:
        mat.params["name_s"] = mat.params["name_s"][-shells:]
        kw = dict(Wc=50.0, tol_E=1e-2, tol_W=1e-2, grid_search="library")
    tr = engine.Transport(mat, 8000.0, 1000.0, s_tilt=60.0, **kw)
    n = 5000
    g = np.random.default_rng(n_bins).standard_normal(1 + n_bins).astype(np.float32)
    J = np.asarray(tr.jacobian(n, seed=3, n_bins=n_bins))
    out = np.asarray(tr.vjp(n, torch.from_numpy(g), seed=3))
    assert J[0, 0] > 0 and np.isfinite(J).all()
    assert abs(J[1:, 0].sum() - J[0, 0]) <= 1e-4 * J[0, 0]
    want, size = g.astype(np.float64) @ J, np.abs(g).astype(np.float64) @ np.abs(J)
    assert (np.abs(out - want) <= 1e-4 * np.maximum(size, np.abs(J).sum() * 1e-3)).all()
