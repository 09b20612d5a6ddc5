"""mcd_scatter_rows: scatter rows put in (electron, step) order on the device
against a sort of the raw rows on the host."""
import ctypes as C

import numpy as np
import pytest
import torch

from mcd import _abi, engine
from mcd._lib import MCDError, check, lib

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tr():
    return engine.Transport("Si", 5000.0, 1000.0, Wc=100.0, s_tilt=40.0, tol_E=1e-2, tol_W=1e-2, max_scatt=70)


@pytest.mark.parametrize("guard", [None, "inline"])
@pytest.mark.parametrize("n,kept,first", [(1, 1, 0), (1025, 1025, 3), (3000, 700, (1 << 32) - 100), (5, 0, 9)])
@pytest.mark.parametrize("fields", [None, ("channel",), ("E_loss", "channel", "x", "step_flags", "config")])
def test_rows_equal_a_host_sort(tr, n, kept, first, fields, guard):
    dev = torch.device("cuda", 0)
    els = torch.empty(n * _abi.ELECTRON_DTYPE.itemsize, dtype=torch.uint8, device=dev)
    cnt = torch.zeros(_abi.NCOUNTERS, dtype=torch.int64, device=dev)
    rows = torch.empty(71 * max(kept, 1) * _abi.SCATTER_DTYPE.itemsize, dtype=torch.uint8, device=dev)
    tr.launch(n, els, cnt, seed=6, first=first, scat_rows=rows, scat_max_electron=first + kept, guard=guard)
    used = int(cnt[_abi.CNT_SCAT_ROWS])
    raw = rows.cpu().numpy()[: used * _abi.SCATTER_DTYPE.itemsize].view(_abi.SCATTER_DTYPE)
    raw = raw[np.lexsort((raw["step"], _abi.row_offsets(raw, first)))]
    got = tr.run(n, seed=6, first=first, scats=True, scat_max_electron=first + kept, scat_fields=fields,
                 guard=guard).scats
    assert len(got) == used
    assert set(got.dtype.names) == set(_abi.SCATTER_DTYPE.names if fields is None else fields + ("electron", "step"))
    for f in got.dtype.names:
        assert got[f].tobytes() == raw[f].tobytes(), f


def test_requests_that_do_not_fit_are_refused(tr):
    ctx = engine.context(0)
    buf = torch.zeros(4096, dtype=torch.uint8, device="cuda")
    need = C.c_size_t(0)

    def call(mask, out, size, n_els=2, rows=buf.data_ptr()):
        check(lib().mcd_scatter_rows(ctx, rows, 8, buf.data_ptr(), n_els, 0, mask, out, size, C.byref(need), None), ctx)

    for mask in (0, 1 << 18):
        with pytest.raises(MCDError, match="field mask"):
            call(mask, None, 0)
    with pytest.raises(MCDError, match="32 bits"):
        call(3, None, 0, n_els=(1 << 32) + 1)
    call(3, None, 0)
    assert need.value == 256 + 2 * 8  # 8 packed rows of 8 bytes, rounded up, and two starts
    with pytest.raises(MCDError, match="output holds"):
        call(3, buf.data_ptr(), need.value - 1)
    with pytest.raises(MCDError, match="NULL rows"):
        call(3, buf.data_ptr(), 4096, rows=None)
