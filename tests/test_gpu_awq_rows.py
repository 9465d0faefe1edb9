"""AutoAWQ linears in place for several rows of x (MFMA on the AWQ words, i4_awq_mm.hip)
against the GEMV that serves the same call without a workspace, and against float64."""
from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

from oracle import i4ref
from tests import _gen
from tests.test_gpu_parity import f_, host, make_x, t_

pytestmark = pytest.mark.gpu
# the output's rounding (half an ulp: 2^-11 / 2^-8 of a value) against the largest value,
# with the fp32 sums' own error far below it
TOL = {"f16": 1e-3, "bf16": 4e-3}
CODE = {"f16": 1, "bf16": 2}


def awq(pkg, dev, rng, N, K, G, xdt, zeros=True):
    """(in-place AWQ QWeight, its float64 rows)."""
    qw, qz, sc = _gen.awq_weight(rng, 1, K, N, G, np.float16 if xdt == "f16" else "bf16")
    if not zeros:
        qz = np.full_like(qz, np.int32(-2004318072))  # zero point 8 in every nibble
    ref = i4ref.awq_dequant(qw, qz, f_(sc), G)[0]
    return pkg.QWeight(t_(qw, dev), t_(sc, dev), t_(qz, dev) if zeros else None, "awq", G, N,
                       K), ref


def gemv_rows(pkg, w, x, xdt, out=torch.float32):
    """The same call without a workspace: the K-complete GEMV, row by row."""
    y = torch.empty(x.shape[0], w.N, dtype=out, device=x.device)
    cw = w.c()
    rc = pkg.lib().i4_linear(x.data_ptr(), CODE[xdt], x.shape[0], ctypes.byref(cw), None,
                             y.data_ptr(), 0 if out == torch.float32 else CODE[xdt], None, 0,
                             torch.cuda.current_stream().cuda_stream)
    assert rc == 0
    return y


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
@pytest.mark.parametrize("G", [32, 64, 128])
@pytest.mark.parametrize("M,N,K", [(24, 2048, 4096), (65, 512, 2048)])
def test_rows_lose_no_precision(pkg, dev, xdt, G, M, N, K):
    """The fp32 result is no further from float64 than the GEMV's (2-norm; a fifth more for
    the two orders of summation).  In bf16 the products carry a bias that cancels, and what
    is left of its rounding must stay below the GEMV's own."""
    rng = np.random.default_rng(M + G)
    w, dq = awq(pkg, dev, rng, N, K, G, xdt)
    x = t_(make_x(rng, (M, K), xdt), dev)
    ref = x.double().cpu().numpy() @ dq.T

    def err(y):
        d = y.double().cpu().numpy() - ref
        return np.linalg.norm(d) / np.linalg.norm(ref)

    got = err(pkg.ops.linear(x, w, out_dtype=torch.float32))
    assert got <= 1.2 * err(gemv_rows(pkg, w, x, xdt)), got


def test_two_streams_share_one_module(pkg, dev):
    """Calls of several rows on two streams at once, each with inputs of its own: the results
    of the same calls one after the other."""
    rng = np.random.default_rng(71)
    w, _ = awq(pkg, dev, rng, 2048, 4096, 128, "f16")
    lin = pkg.PackedLinear.from_qweight(w, repack=False)
    xs = [[t_(make_x(rng, (rows, 4096), "f16"), dev) for rows in (24, 9, 31, 24)]
          for _ in range(2)]
    want = [[lin(x).clone() for x in side] for side in xs]
    torch.cuda.synchronize()
    streams = [torch.cuda.Stream() for _ in xs]
    got = [[], []]
    for _ in range(30):
        for i, s in enumerate(streams):
            with torch.cuda.stream(s):
                got[i] += [lin(x) for x in xs[i]]
    torch.cuda.synchronize()
    for i in range(2):
        for n, y in enumerate(got[i]):
            assert torch.equal(y, want[i][n % 4])


@pytest.mark.parametrize("xdt,G,zeros", [("f16", 128, True), ("bf16", 128, True),
                                         ("bf16", 64, False), ("f16", 32, False)])
@pytest.mark.parametrize("N,K", [(512, 2048), (1024, 2048), (2048, 1024), (768, 4096)])
def test_few_rows_on_either_path(pkg, dev, xdt, G, zeros, N, K):
    """3..8 rows, on both sides of the line between the GEMV and MFMA, with and without zero
    points, K ranges that end inside a group: against float64, and by which memory of the
    caller's workspace a call writes (MFMA: every fp32 partial behind the GEMV's pairs, and
    not the status word; the GEMV: none of them)."""
    lb = pkg.lib()
    rng = np.random.default_rng(N + G)
    w, dq = awq(pkg, dev, rng, N, K, G, xdt, zeros)
    cw = w.c()
    size = lambda M: lb.i4_linear_workspace_bytes(ctypes.byref(cw), M)
    bias = t_(make_x(rng, (N,), xdt), dev)
    took = set()
    for M in (3, 4, 5, 6, 7, 8):
        x = t_(make_x(rng, (M, K), xdt), dev)
        mm = bool(lb.i4_linear_awq_mfma(ctypes.byref(cw), M))
        took.add(mm)
        nbytes = max(size(M), 256)
        ws = torch.zeros(nbytes, dtype=torch.uint8, device=dev)
        head = max([256] + [lb.i4_dq_gemv_workspace_bytes(ctypes.byref(cw), r)
                            for r in range(1, 9) if not lb.i4_linear_awq_mfma(
                                ctypes.byref(cw), r)])
        if mm:
            assert (nbytes - head) % (M * N * 4) == 0 and nbytes > head
            ws[head:].view(torch.int32).fill_(0x7FC0DEAD)  # a NaN no sum produces
        y = torch.empty(M, N, dtype=x.dtype, device=dev)
        rc = lb.i4_linear(x.data_ptr(), CODE[xdt], M, ctypes.byref(cw), bias.data_ptr(),
                          y.data_ptr(), CODE[xdt], ws.data_ptr() if nbytes else None, nbytes,
                          torch.cuda.current_stream().cuda_stream)
        assert rc == 0
        ref = x.double().cpu().numpy() @ dq.T + bias.double().cpu().numpy()
        assert i4ref.rel_err(y.double().cpu().numpy(), ref) <= TOL[xdt]
        assert int(ws[:4].view(torch.int32)[0]) == 0
        if mm:
            assert not bool((ws[head:].view(torch.int32) == 0x7FC0DEAD).any())
            assert not bool(ws[4:head].any())
    assert False in took  # 3 rows: the GEMV


@pytest.mark.parametrize("xdt", ["f16", "bf16"])
def test_nonfinite_rows_stay_apart(pkg, dev, xdt):
    """Infinities and NaN in some rows of x reach those rows' outputs only."""
    rng = np.random.default_rng(79)
    w, _ = awq(pkg, dev, rng, 2048, 4096, 128, xdt)
    x = t_(make_x(rng, (37, 4096), xdt), dev)
    clean = pkg.ops.linear(x, w)
    bad = {0: float("inf"), 15: float("nan"), 16: float("-inf"), 36: float("nan")}
    for r, v in bad.items():
        x[r, 37 * r % 4096] = v
    got = pkg.ops.linear(x, w)
    for r in range(37):
        if r in bad:
            assert not bool(torch.isfinite(got[r]).any())
        else:
            assert torch.equal(got[r], clean[r])
