"""The Newton-Schulz plan's buffers and tables on the CPU, the launches recorded."""

import numpy as np
import pytest
import torch

from apexw_amd import _lib, muon


class _Lib:
    def __init__(self, real):
        self.real, self.tables = real, []

    def __getattr__(self, name):
        return getattr(self.real, name)

    def apexw_muon_prepare_grouped(self, items, *rest):
        self.tables.append(items)
        return 0


@pytest.fixture
def lib(monkeypatch):
    rec = _Lib(_lib.load())
    monkeypatch.setattr(_lib, "load", lambda: rec)
    monkeypatch.setattr(_lib, "cus_per_queue", lambda device: 32)      # the chip's 256 CUs
    monkeypatch.setattr(torch.Tensor, "pin_memory", lambda self: self)
    return rec


def _plan(m, n, batch, steps=5):
    ws = muon.NSWorkspace(m, n, batch, torch.device("cpu"))
    return ws, muon.NSPlan([ws], [steps], torch.device("cpu"))


def _items(ws, m, n):
    return np.array([(1 << 20, 1 << 21, x, 0, part, m, n, ws.np_, ws.mp, 0.95, 0.05, _lib.F32, ws.layout, 1, 0)
                     for x, part in ws.rows], dtype=_lib.MUON_ITEM_DTYPE)


@pytest.mark.parametrize("m,n,batch,steps,reads", [(768, 3072, 24, 5, False),      # [K x N] rows
                                                   (768, 3072, 24, 0, False),      # no product
                                                   (1792, 1792, 14, 5, True),      # K beyond NN_MAX_K
                                                   (500, 500, 2, 5, True)])        # 128 x 128 tiles
def test_x_transposed_is_kept_only_where_a_product_reads_it(lib, m, n, batch, steps, reads):
    ws, plan = _plan(m, n, batch, steps)
    items = _items(ws, m, n)
    plan.prepare(0, items, 1.0)
    assert (ws._xt is not None) == reads
    want = [t.data_ptr() for t in ws.xt[0]] if reads else [0] * batch
    assert items["xt"].tolist() == want
    if reads:
        assert not any(bool(t.any()) for t in ws.xt)      # the padding starts, and stays, zero


def test_item_table_is_not_shared_between_streams(lib):
    ws, plan = _plan(64, 64, 1)
    keep = []
    for stream in (1, 1, 2, 2):
        plan.prepare(stream, _items(ws, 64, 64), 1.0)
        keep.append(plan._prepared)
    assert lib.tables[0] == lib.tables[1] and lib.tables[2] == lib.tables[3]
    assert lib.tables[2] != lib.tables[1]
