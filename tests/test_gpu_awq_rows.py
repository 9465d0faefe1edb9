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
DT = {"f16": torch.float16, "bf16": torch.bfloat16}
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
