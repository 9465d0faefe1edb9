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


def _mm_rows(pkg, N, K, G, rows):
    import ctypes

    w = awq_linear(pkg, N, K, G).w.c()
    return [M for M in rows if pkg.lib().i4_linear_awq_mfma(ctypes.byref(w), M)]


@pytest.mark.parametrize("N,K,G,first", [
    # the K-complete GEMV was measured faster below: M N K under 8 M, 20 M below 256 columns
    (128, 256, 128, None), (128, 2048, 32, 80), (64, 2048, 128, None), (512, 768, 128, 22),
    (2048, 256, 32, 16), (1024, 256, 64, 32),
    # against the split GEMV: 112 slices to hand over, or M N K of 24 / 12 / 8 M
    (2048, 4096, 128, 4), (2048, 2048, 128, 6), (4096, 1024, 128, 6), (512, 2048, 128, 7),
    (2048, 2048, 64, 4), (2048, 1024, 32, 4), (4096, 768, 64, 4), (64, 8192, 128, 4),
])
def test_rows_take_mfma_where_it_was_measured_faster(pkg, N, K, G, first):
    """The first row count on MFMA; every later one too, up to 8 rows (split GEMV) and from 9
    (K-complete GEMV) apart."""
    rows = _mm_rows(pkg, N, K, G, range(1, 160))
    if first is None:
        assert not rows
    else:
        assert rows[0] == first
        few, many = [r for r in rows if r <= 8], [r for r in rows if r > 8]
        for part, last in ((few, 8), (many, 159)):
            assert not part or part == list(range(part[0], last + 1))


@pytest.mark.parametrize("N,K,M,gemv_rows,ksplit", [
    (2048, 4096, 24, 3, 16), (512, 2048, 24, 6, 16), (4096, 2048, 33, 3, 4),
    (2048, 256, 64, 5, 2), (768, 768, 24, 8, 6),
])
def test_partials_start_behind_the_weights_own_pairs(pkg, N, K, M, gemv_rows, ksplit):
    """The workspace of M rows: what the split GEMV of up to gemv_rows rows of this weight
    uses (at least the 256-byte header), then ksplit partials of M x N fp32."""
    import ctypes

    w = awq_linear(pkg, N, K).w.c()
    lb = pkg.lib()
    head = max([256] + [lb.i4_dq_gemv_workspace_bytes(ctypes.byref(w), r)
                        for r in range(1, gemv_rows + 1)])
    assert lb.i4_linear_workspace_bytes(ctypes.byref(w), M) == head + ksplit * M * N * 4
