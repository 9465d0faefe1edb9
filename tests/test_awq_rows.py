"""Host side of AutoAWQ linears in place for several rows of x: which memory a call hands to
the library (i4_linear itself is stubbed; the workspace sizes are the library's)."""
from __future__ import annotations

import pytest
import torch


class _Stub:
    """The library with i4_linear recorded instead of launched."""

    def __init__(self, real):
        self.real, self.calls = real, []

    def __getattr__(self, name):
        return getattr(self.real, name)

    def i4_linear(self, x, xt, M, w, bias, y, yt, ws, ws_bytes, stream):
        self.calls.append((M, ws, ws_bytes))
        return 0


@pytest.fixture
def stub(pkg, monkeypatch):
    lib = _Stub(pkg.lib())
    monkeypatch.setattr(pkg._lib, "lib", lambda: lib)
    monkeypatch.setattr(pkg._lib, "require_device", lambda *ts: torch.device("cpu"))
    monkeypatch.setattr(pkg._lib, "stream", lambda device: 0)
    return lib


def awq_linear(pkg, N, K, G=128):
    w = pkg.QWeight(torch.zeros(1, K, N // 8, dtype=torch.int32),
                    torch.ones(1, K // G, N, dtype=torch.float16),
                    torch.zeros(1, K // G, N // 8, dtype=torch.int32), "awq", G, N, K)
    return pkg.PackedLinear.from_qweight(w, repack=False)


def test_rows_leave_the_kept_workspace_alone(pkg, stub):
    """One row takes the module's kept split-K workspace; calls of more rows (whose partials
    live for one call) neither replace nor use it, so a graph captured on the one-row call
    keeps its buffer and calls on two streams share nothing."""
    lin = awq_linear(pkg, 2048, 4096)
    x = lambda rows: torch.zeros(rows, 4096, dtype=torch.float16)
    lin(x(1))
    kept = lin.workspace.buf
    lo, hi = kept.data_ptr(), kept.data_ptr() + kept.numel()
    assert stub.calls[-1][1] == lo
    for rows in (24, 256, 33, 4):
        lin(x(rows))
        M, ws, nbytes = stub.calls[-1]
        assert M == rows and lin.workspace.buf is kept
        assert ws is None or ws + nbytes <= lo or ws >= hi
    lin(x(1))
    assert stub.calls[-1][1] == lo
