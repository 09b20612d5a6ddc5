"""Table kernels.  CDF rows (k_build_cdf: a wavefront to a row, tiles of 256
loss bins) at the edges of its tiles, against FP64 sums in numpy; the kinds of the
pick table's cells (k_pick_cells, k_pick_check)."""
import numpy as np
import pytest

from conftest import gpu_available
from mcd import _abi, engine
from mcd.material import Material
from mcd.tables import gryz_grid, moller_grid

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]

PI_E4 = 6.51408491409531e-14  # pi e^4 [eV^2 cm^2]; cancels in the quotient


def _rows(g, Ef, kind):
    """Running sums over their total, one bin after the other (computeBlock, probTables.py:415-462)."""
    out = np.full((len(g.Es), len(g.Ws) - 1), 2.0)
    W = g.Ws.astype(np.float64)
    for i, E32 in enumerate(g.Es):
        E = float(E32)
        valid = ~(g.Ws[1:] > (E32 - np.float32(Ef)) * np.float32(0.5))
        with np.errstate(all="ignore"):
            eps, epsB = W / E, g.Eb / E
            if kind == "moller":
                f = PI_E4 * (1 / eps**2 + 1 / (1 - eps)**2 - 1 / (eps * (1 - eps))) / E**3
                f[~(eps < 1)] = 0
            else:
                f = (PI_E4 * eps * (1 + epsB)**-1.5 * (1 - eps)**(epsB / (epsB + eps)) *
                     ((1 - epsB) + 4 * epsB * np.log(2.7 + np.sqrt((1 - eps) / epsB)) / (3 * eps)) / W**3)
                f[~((eps < 1) & (epsB < 1))] = 0
        m = int(valid.sum())
        t = np.cumsum((W[1:m + 1] - W[:m]) * (f[:m] + f[1:m + 1]) / 2)
        out[i, :m] = t / t[-1] if m else 0
    return out, np.array([int((r < 2).sum()) for r in out])


# float32 of a quotient that is right to 1e-12 (the shared sums): half an ulp of 1, and as much where it straddles
@pytest.mark.parametrize("nE,nW", [(2, 2), (3, 3), (4, 64), (5, 65), (7, 66), (9, 256), (6, 257), (6, 258), (13, 514), (3, 1500)])
def test_cdf_rows_equal_sequential_fp64_sums(nE, nW):
    cu = Material("Cu")
    gm, gg = moller_grid(cu, 20000.0, 1000.0, 50.0), gryz_grid(cu, 20000.0, 1000.0)
    for g in (gm, gg):
        g.Es = np.linspace(1000.0, 20000.0, nE).astype(np.float32)
        # up to past the largest loss of the rows: whole, part and no valid bins
        g.Ws = np.geomspace(g.Wmin, 12000.0, nW).astype(np.float32)
    for prec, tol in ((_abi.PREC_FP64, 1.2e-7), (_abi.PREC_FP32, 1.2e-7 * max(nW, 64))):
        tr = engine.Transport("Cu", 20000.0, 1000.0, Wc=50.0, grids=(gm, gg), table_precision=prec)
        for q, g, kind in ((0, gm, "moller"), (1, gg, "gryz")):
            ref, m = _rows(g, tr.mat.fermi_e, kind)
            got = tr.cdf(q)
            for i in range(nE):
                assert np.abs(got[i, :m[i]] - ref[i, :m[i]]).max(initial=0.0) <= tol, (q, prec, i)
            masked = [set(np.unique(got[i, m[i]:])) for i in range(nE)]
            assert all(len(v) <= 1 for v in masked)


# Cell kinds and guard bands as a classification of the node orders and check errors on the host gave them
# (swapped neighbours, exact cells at thresholds and in coarse tables); the band within float32's last digit
@pytest.mark.parametrize("kw,nodes,swaps,exact,delta", [
    (dict(material="Al", E0=5000.0, Emin=80.0, Wc=20.0), 16, 1, 11, 0.00017833914898801595),
    (dict(material="Al", E0=5000.0, Emin=80.0, Wc=20.0), 512, 1, 0, 1.1658748917398043e-06),
    (dict(material="Si", E0=3000.0, Emin=105.0, Wc=100.0, elastic="Ruth_nigram"), 17, 2, 4, 0.00015346590953413397),
    (dict(material="Si", E0=3000.0, Emin=105.0, Wc=100.0, elastic="Ruth_nigram"), 512, 2, 11, 0.0001922775263665244),
    (dict(material="Cu", E0=1500.0, Emin=60.0, Wc=50.0), 100, 2, 10, 0.00018746251589618623),
    (dict(material="Au", E0=30000.0, Emin=90.0, Wc=20.0), 16, 2, 4, 0.00016507641703356057),
    (dict(material="Au", E0=30000.0, Emin=90.0, Wc=20.0), 100, 4, 0, 1.8642254872247577e-05),
], ids=str)
def test_pick_table_cells_and_guard_band(kw, nodes, swaps, exact, delta):
    info = engine.Transport(tol_E=5e-2, tol_W=5e-2, grid_search="library", pick_nodes=nodes, **kw).pick_info()
    assert (info["n_nodes"], info["swap_cells"], info["exact_cells"]) == (nodes, swaps, exact)
    assert abs(info["delta"] - delta) <= 2.4e-7
