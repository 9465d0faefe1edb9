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
    monkeypatch.setattr(pkg.ops, "_test_capture", False, raising=False)
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


def test_large_moe_calls_keep_no_large_workspace(pkg, monkeypatch):
    """A call of thousands of tokens takes its scratch for the call: the module's workspace
    keeps the size of a 1024-token call, or the status word's, however many layers ran."""
    lib = pkg.lib()
    calls = []

    class Stub:
        def __getattr__(self, name):
            return getattr(lib, name)

        def i4_moe_forward(self, *a):
            calls.append((a[2], a[11], a[12], None))
            return 0

        def i4_moe_forward_status(self, *a):
            calls.append((a[2], a[11], a[12], a[13]))
            return 0

    monkeypatch.setattr(pkg._lib, "lib", lambda: Stub())
    monkeypatch.setattr(pkg._lib, "require_device", lambda *ts: CPU)
    monkeypatch.setattr(pkg._lib, "stream", lambda device: 0)
    H, I, E, k = 256, 128, 24, 8
    w = lambda n, kk: pkg.QWeight(torch.zeros(E, n // 16, kk // 128, 16, 16, dtype=torch.int32),
                                  torch.ones(E, n // 16, kk // 32, 16, dtype=torch.float16),
                                  None, "tile", 32, n, kk)
    gu, dn = w(2 * I, H), w(H, I)
    router = torch.zeros(E, H, dtype=torch.float16)
    ws = pkg.Workspace()
    run = lambda T: pkg.moe_forward(torch.zeros(T, H, dtype=torch.float16), gu, dn, k,
                                    router_w=router, workspace=ws)
    least = lib.i4_moe_workspace_bytes(1024, H, I, E, k)
    off = lib.i4_moe_status_offset(1, H, I, E, k)
    run(3000)
    assert ws.buf.numel() == off + 4
    assert calls[-1][2] == lib.i4_moe_workspace_bytes(3000, H, I, E, k) > least
    assert calls[-1][3] == ws.buf.data_ptr() + off
    run(1024)
    kept = ws.buf
    assert kept.numel() == least and calls[-1][1] == kept.data_ptr()
    run(4096)
    assert ws.buf is kept and calls[-1][1] != kept.data_ptr()
    assert calls[-1][3] == kept.data_ptr() + off
