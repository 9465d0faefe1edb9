"""ops.Workspace: a buffer that a captured graph writes to outlives the workspace's growth."""
from __future__ import annotations

import weakref

import pytest
import torch

CPU = torch.device("cpu")


@pytest.fixture
def ops(pkg, monkeypatch):
    monkeypatch.setattr(pkg.ops, "_capturing", lambda device: pkg.ops._test_capture,
                        raising=False)
    pkg.ops._test_capture = False
    return pkg.ops


def test_growth_keeps_a_captured_buffer(ops):
    """Warm up, capture, then ask for more: the captured buffer stays alive, and does so once
    however often it was handed out."""
    ws = ops.Workspace()
    first = ws.get(1000, CPU)
    ops._test_capture = True
    assert ws.get(1000, CPU) is first
    assert ws.get(500, CPU) is first
    ops._test_capture = False
    alive = weakref.ref(first)
    addr = first.data_ptr()
    del first
    assert ws.get(1001, CPU).numel() >= 1001
    assert alive() is not None and [b.data_ptr() for b in ws.kept] == [addr]


def test_growth_without_capture_frees(ops):
    ws = ops.Workspace()
    alive = weakref.ref(ws.get(1000, CPU))
    ws.get(4000, CPU)
    assert alive() is None and not ws.kept and ws.buf.numel() == 4000


def test_kept_buffers_are_bounded(ops):
    """Captures at ever larger sizes: the kept buffers add up to at most the one in use."""
    ws = ops.Workspace()
    for n in range(1000, 9000, 100):
        ops._test_capture = True
        ws.get(n, CPU)
        ops._test_capture = False
        ws.get(n + 1, CPU)
    assert sum(b.numel() for b in ws.kept) <= ws.buf.numel() <= 4 * 9000


def test_status_of_a_kept_buffer(ops, monkeypatch):
    """A give-up that a replay reports in a kept buffer is still read."""
    monkeypatch.setattr(torch.cuda, "synchronize", lambda device=None: None)
    ws = ops.Workspace()
    ops._test_capture = True
    first = ws.get(512, CPU, zeroed=True)
    ops._test_capture = False
    ws.get(2048, CPU, zeroed=True)
    assert ops.gemv_status(ws) == 0
    first[:4].view(torch.int32).fill_(-10)
    assert ops.gemv_status(ws) == -10
