"""Graphs of small calls replayed after larger eager calls of the same module: the replay
writes only to memory that still is the module's, and gives the eager result."""
from __future__ import annotations

import numpy as np
import pytest
import torch

from tests.test_gpu_awq_rows import awq
from tests.test_gpu_parity import _awq_moe, make_x, t_

pytestmark = pytest.mark.gpu


def replay_after_larger(module, small, larger, workspace):
    """Capture module(small), run module(l) for l in larger, fill whatever the allocator now
    holds free, then replay with new inputs and eager work in between."""
    static = small[0].clone()
    want = [module(x).clone() for x in small]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        module(static)
    torch.cuda.current_stream().wait_stream(side)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = module(static)
    held = 1 << 23 if workspace.buf is None else workspace.buf.numel()
    for x in larger:
        module(x)
    torch.cuda.synchronize()
    fill = [torch.full((held // n,), 0x5A, dtype=torch.uint8, device=static.device)
            for n in (1, 1, 2, 4, 8)]
    for x, w in zip(small * 2, want * 2):
        static.copy_(x)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, w)
        assert torch.equal(module(x), w)  # eager work between the replays
    assert all(bool((f == 0x5A).all()) for f in fill)


@pytest.mark.parametrize("T", [1, 5])
def test_moe_graph_after_larger_calls(pkg, dev, T):
    rng = np.random.default_rng(61 + T)
    moe, _, _, _ = _awq_moe(pkg, dev, rng, E=32)
    small = [t_(make_x(rng, (T, 2048), "f16"), dev) for _ in range(3)]
    larger = [t_(make_x(rng, (n, 2048), "f16"), dev) for n in (40, 300)]
    replay_after_larger(moe, small, larger, moe.workspace)
    assert pkg.moe_status(moe.workspace, T, 2048, moe.down.K, 32, moe.top_k) == 0


@pytest.mark.parametrize("rows", [1, 4, 12])
@pytest.mark.parametrize("N,K", [(2048, 4096), (512, 2048)])
def test_awq_linear_graph_after_larger_calls(pkg, dev, rows, N, K):
    """One row (the split-K GEMV on the module's workspace) and several rows (partials of the
    call, here of the graph)."""
    rng = np.random.default_rng(67 + rows)
    w, _ = awq(pkg, dev, rng, N, K, 128, "f16")
    lin = pkg.PackedLinear.from_qweight(w, repack=False)
    small = [t_(make_x(rng, (rows, K), "f16"), dev) for _ in range(3)]
    larger = [t_(make_x(rng, (n, K), "f16"), dev) for n in (24, 256)]
    replay_after_larger(lin, small, larger, lin.workspace)
    assert pkg.ops.gemv_status(lin.workspace) == 0


def test_moe_prompt_after_capture(pkg, dev):
    """A captured call of 70 tokens, then prompts beyond 1024: the workspace stays."""
    rng = np.random.default_rng(73)
    moe, _, _, _ = _awq_moe(pkg, dev, rng, E=24, H=256, I=128, G=32)
    small = [t_(make_x(rng, (70, 256), "f16"), dev) for _ in range(3)]
    larger = [t_(make_x(rng, (n, 256), "f16"), dev) for n in (1500, 4100)]
    replay_after_larger(moe, small, larger, moe.workspace)
    assert moe.workspace.buf.numel() == pkg.lib().i4_moe_workspace_bytes(70, 256, 128, 24, 8)
    assert pkg.moe_status(moe.workspace, 4100, 256, 128, 24, 8) == 0
