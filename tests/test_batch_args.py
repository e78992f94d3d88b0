"""CPU test of batch.run_batch's arguments: every box has its own entry of
``ws``, and a list that is too short is refused before anything is launched
(the boxes' records would otherwise stay empty)."""
import numpy as np
import pytest
import torch

from pyspectrum_amd import batch as B


class _Ctx:
    def __init__(self):
        self.calls = []

    def call(self, name, *args):
        self.calls.append((name, args))


@pytest.fixture
def host_only(monkeypatch):
    """run_batch with its device and counts replaced by host stand-ins."""
    monkeypatch.setattr(B.P, "_device", lambda d: torch.device("cpu"))
    monkeypatch.setattr(B.P, "_counts_Bk123", lambda **kw: None)
    monkeypatch.setattr(B.P, "_tri_counts", lambda c, ijl, N: np.ones(len(ijl)))
    monkeypatch.setattr(B.L, "triangles", lambda *a: np.ones((1, 3), dtype=np.int32))


def _run(ctx, ws):
    xyzs = [torch.zeros((3, n)) for n in (5, 7)]
    B.run_batch(ctx, xyzs, ws, [10.0, 20.0], 16, 1, 1, 1, "fp32", 0, half=torch.zeros(1))


def test_short_weight_list_is_refused(host_only):
    ctx = _Ctx()
    with pytest.raises(IndexError):
        _run(ctx, [np.ones(5)])
    assert ctx.calls == []


def test_every_box_gets_its_weights(host_only):
    ctx = _Ctx()
    _run(ctx, [None, np.full(7, 2.0)])
    boxes = ctx.calls[0][1][1]
    assert [(b.np, b.sumw, bool(b.w)) for b in boxes] == [(5, 5.0, False), (7, 14.0, True)]
