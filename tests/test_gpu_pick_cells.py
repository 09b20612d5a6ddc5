"""Pick tables with cells a few ulp of ln E wide: check points fall into
neighbouring cells, whose kinds stay as they are until every point is checked."""
import pytest

from conftest import gpu_available
from mcd import engine

pytestmark = [pytest.mark.gpu, pytest.mark.skipif(not gpu_available(), reason="no GPU")]


# a classification of check points on the host gave these guard bands; the band within float32's last digit
@pytest.mark.parametrize("kw,nodes,delta", [
    (dict(material="Cu", E0=1100.0, Emin=1000.0, Wc=50.0), 8192, 3.5007550991394965e-07),
    (dict(material="Cu", E0=1001.0, Emin=1000.0, Wc=50.0), 512, 3.318673122976179e-07),
    (dict(material="Au", E0=30000.0, Emin=29900.0, Wc=20.0), 8192, 2.73022777719234e-07),
], ids=str)
def test_narrow_cells(kw, nodes, delta):
    infos = [engine.Transport(tol_E=5e-2, tol_W=5e-2, grid_search="library", pick_nodes=nodes, **kw).pick_info()
             for _ in range(4)]
    assert all(i == infos[0] for i in infos)
    assert (infos[0]["swap_cells"], infos[0]["exact_cells"]) == (0, 0)
    assert abs(infos[0]["delta"] - delta) <= 2.4e-7
