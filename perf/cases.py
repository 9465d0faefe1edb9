"""Workloads of this framework, each one pass through its public entry points.

The families are the work a duplex session has the library do, at the sizes of the Thinker
(hidden 2048, 128 int4 experts, top-8, FFN 768, 32 query and 4 key/value heads of 128) and
of the Talker (hidden 1024, 128 16-bit or int8 experts, top-6, FFN 384, shared expert 768):

  linear   PackedLinear: one int4 projection, from one token (a decode frame) to a prompt of
           thousands; compressed-tensors rows ("ct", the checkpoint's format, bf16, groups of
           32) or AutoAWQ packing read in place ("awq", fp16, groups of 128, zero points)
  moe      FusedPackedMoE with its pre-MoE RMSNorm and residual: a few concurrent sessions,
           prompt chunks, whole prompts; the routing may be skewed towards popular experts
  stack    moe_stack: one decode token through the layers' MoE blocks
  decoder  ThinkerDecoder.step: one decode token through whole decoder layers with a KV cache
  talker   FusedMoE with residual: 16-bit or int8 experts, a few tokens up to a prompt
  chain    one Talker decode token through its blocks, captured once in a graph and replayed
           per token, as the per-frame loop runs it

Weights are random of the real formats; inputs are made from the seed alone, on the GPU.
"""
from __future__ import annotations

import importlib.util
import math
import sys
from pathlib import Path
from types import SimpleNamespace

import torch

ROOT = Path(__file__).resolve().parents[1]
DEV = "cuda"
DT = {"bf16": torch.bfloat16, "fp16": torch.float16}
E, H, I, TOPK = 128, 2048, 768, 8            # Thinker MoE block
NH, NKV, HD, THETA = 32, 4, 128, 1_000_000.0  # Thinker attention
TE, TH, TI, TIS, TK = 128, 1024, 384, 768, 6  # Talker MoE block
EPS = 1e-6
# projections of a Thinker layer: q, k / v, o, fused q|k|v, and a single expert row block
SHAPES = {"q": (2048, 4096), "kv": (2048, 512), "o": (4096, 2048), "qkv": (2048, 5120),
          "expert": (2048, 768)}


def _package():
    name = "qwen3_omni_duplex_amd"
    if name not in sys.modules:
        root = ROOT / "qwen3-omni-duplex_amd"
        spec = importlib.util.spec_from_file_location(name, root / "__init__.py",
                                                      submodule_search_locations=[str(root)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules[name] = mod
        spec.loader.exec_module(mod)
    return sys.modules[name]


def listed():
    return [
        # one expert-sized projection of one decode token: the smallest call there is
        {"name": "linear_token", "family": "linear", "fmt": "ct", "shape": "expert", "rows": 1},
        # the output projection of 24 sessions decoding together, AutoAWQ weights in place
        {"name": "linear_awq_batch", "family": "linear", "fmt": "awq", "shape": "o", "rows": 24},
        # q|k|v of a 1500-token prompt
        {"name": "linear_prompt", "family": "linear", "fmt": "ct", "shape": "qkv", "rows": 1500},
        # the clock path's MoE layers for one 80 ms frame
        {"name": "stack_token", "family": "stack", "fmt": "awq", "layers": 24},
        # the clock path's whole Thinker[0:24] step, 1024 positions in the cache
        {"name": "decoder_token", "family": "decoder", "fmt": "ct", "layers": 24, "pos": 1024},
        # 13 sessions' tokens through one MoE block
        {"name": "moe_batch", "family": "moe", "fmt": "awq", "rows": 13, "skew": 0.0},
        # a 512-token prompt chunk with popular experts
        {"name": "moe_chunk", "family": "moe", "fmt": "awq", "rows": 512, "skew": 1.0},
        # a whole 3001-token prompt in the checkpoint's own format
        {"name": "moe_prompt", "family": "moe", "fmt": "ct", "rows": 3001, "skew": 0.5},
        # one Talker token through its 20 blocks
        {"name": "talker_token", "family": "chain", "q8": False, "layers": 20},
        # 37 Talker tokens (a short segment) on int8 experts
        {"name": "talker_q8_segment", "family": "talker", "q8": True, "rows": 37},
        # 150 tokens of Talker context on bf16 experts
        {"name": "talker_segment", "family": "talker", "q8": False, "rows": 150},
        # a 700-token Talker prompt
        {"name": "talker_prompt", "family": "talker", "q8": False, "rows": 700},
    ]


def draw(rng):
    def log_int(lo, hi):
        return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))

    family = rng.choice(["linear", "linear", "moe", "moe", "talker", "talker", "stack",
                         "decoder", "chain"])
    if family == "linear":
        fmt = rng.choice(["ct", "awq"])
        return {"family": family, "fmt": fmt, "shape": rng.choice(sorted(SHAPES)),
                "rows": log_int(1, 2048 if fmt == "ct" else 256)}
    if family == "moe":
        return {"family": family, "fmt": rng.choice(["ct", "awq"]), "rows": log_int(2, 3000),
                "skew": round(rng.uniform(0.0, 1.0), 2)}
    if family == "talker":
        return {"family": family, "q8": rng.random() < 0.5, "rows": log_int(2, 700)}
    if family == "stack":
        return {"family": family, "fmt": rng.choice(["ct", "awq"]), "layers": rng.randint(2, 24)}
    if family == "decoder":
        return {"family": family, "fmt": "ct", "layers": rng.randint(2, 12),
                "pos": log_int(3, 4000)}
    return {"family": "chain", "q8": rng.random() < 0.5, "layers": rng.randint(2, 20)}


# ------------------------------------------------------------------------------- inputs
def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g, *shape, sd=1.0, dt=torch.float32):
    return (torch.randn(*shape, device=DEV, generator=g) * sd).to(dt)


def _words(g, *shape):
    return torch.randint(-2**31, 2**31, shape, dtype=torch.int32, device=DEV, generator=g)


def _vec(g, n, dt):
    return (torch.rand(n, device=DEV, generator=g) * 0.4 + 0.8).to(dt)


def _fmt(case):
    """(dtype, group, zero points) of a case's weight format."""
    return (torch.bfloat16, 32, False) if case["fmt"] == "ct" else (torch.float16, 128, True)


def _weight(g, e, n, k, case, gain=1.0):
    """Random CT rows: packed [e, n, k/8], scale [e, n, groups], zeros (packed) or None.
    Nibbles are uniform around the zero point; the values' deviation is gain / sqrt(k)."""
    dt, group, zp = _fmt(case)
    ng = k // group
    base = gain / math.sqrt(k) / (6.5 if zp else 4.6)
    scale = ((torch.rand(e, n, ng, device=DEV, generator=g) + 0.5) * base).to(dt)
    return (_words(g, e, n, k // 8), scale, _words(g, e, n, -(-ng // 8)) if zp else None, group,
            n, k)


def _q(w):
    packed, scale, zeros, group, n, k = w
    return _package().QWeight(packed, scale, zeros, "ct", group, n, k)


def _moe_parts(g, case):
    dt, _, _ = _fmt(case)
    return SimpleNamespace(
        gu=_weight(g, E, 2 * I, H, case), dn=_weight(g, E, H, I, case),
        rw=_randn(g, E, H, sd=0.04, dt=dt), nw=_vec(g, H, dt))


def _moe_module(p):
    return _package().FusedPackedMoE.from_stacked(_q(p.gu), _q(p.dn), p.rw, TOPK,
                                                  norm_weight=p.nw, norm_eps=EPS)


def _popular(g, p, skew, rows, dt):
    """Rows whose router logits lean towards popular experts: every row has a common part,
    along which expert e's router row has a weight that falls with its rank."""
    x = torch.randn(rows, H, device=DEV, generator=g)
    m = torch.randn(H, device=DEV, generator=g)
    m /= m.norm()
    rank = torch.argsort(torch.rand(E, device=DEV, generator=g)).float()
    lean = -torch.log1p(rank) * skew
    p.rw = (p.rw.float() + torch.outer(lean - lean.mean(), m) / math.sqrt(H) * 2).to(dt)
    return (x + m * (0.5 * math.sqrt(H))).to(dt)


def _talker_parts(g, dt, gain=1.0):
    """One Talker block; gain scales gate and up (a chain without norms between its blocks
    needs less than 1 to keep the residual stream's size)."""
    r = lambda *s, sd: _randn(g, *s, sd=sd, dt=dt)  # noqa: E731
    return SimpleNamespace(gu=r(TE, 2 * TI, TH, sd=gain * TH ** -0.5),
                           dn=r(TE, TH, TI, sd=TI ** -0.5), rw=r(TE, TH, sd=0.05),
                           sgu=r(2 * TIS, TH, sd=gain * TH ** -0.5),
                           sdn=r(TH, TIS, sd=TIS ** -0.5), sgw=r(TH, sd=0.05))


class _Holder(torch.nn.Module):
    def __init__(self, **kw):
        super().__init__()
        for k, v in kw.items():
            setattr(self, k, torch.nn.Parameter(v, requires_grad=False)
                    if isinstance(v, torch.Tensor) else v)


def _talker_module(p, q8):
    """FusedMoE built from a block of the stacked-parameter form."""
    block = _Holder(
        gate=_Holder(weight=p.rw), top_k=TK, norm_topk_prob=True,
        experts=_Holder(gate_up_proj=p.gu, down_proj=p.dn),
        shared_expert=_Holder(gate_proj=_Holder(weight=p.sgu[:TIS]),
                              up_proj=_Holder(weight=p.sgu[TIS:]),
                              down_proj=_Holder(weight=p.sdn)),
        shared_expert_gate=_Holder(weight=p.sgw.view(1, -1)))
    return _package().FusedMoE(block, q8=q8)


def _linear_parts(g, case):
    """Weight of a linear case: CT rows, or AutoAWQ words [k, n/8], scales and zeros."""
    k, n = SHAPES[case["shape"]]
    if case["fmt"] == "ct":
        return _weight(g, 1, n, k, case)
    ng = k // 128
    scale = ((torch.rand(1, ng, n, device=DEV, generator=g) + 0.5)
             / (6.5 * math.sqrt(k))).half()
    return _words(g, 1, k, n // 8), scale, _words(g, 1, ng, n // 8), 128, n, k


def _inv_freq():
    return 1.0 / (THETA ** (torch.arange(0, HD, 2, dtype=torch.float) / HD))


def _decoder_parts(g, case):
    dt = torch.bfloat16
    layers = []
    for _ in range(case["layers"]):
        p = _moe_parts(g, case)
        p.wq = _weight(g, 1, NH * HD, H, case)
        p.wk = _weight(g, 1, NKV * HD, H, case)
        p.wv = _weight(g, 1, NKV * HD, H, case)
        p.wo = _weight(g, 1, H, NH * HD, case)
        p.qn, p.kn, p.inn = _vec(g, HD, dt), _vec(g, HD, dt), _vec(g, H, dt)
        p.k = _randn(g, NKV, case["pos"], HD, dt=dt)
        p.v = _randn(g, NKV, case["pos"], HD, dt=dt)
        layers.append(p)
    return layers


def _make(case, seed):
    """The random parts of a case, in a fixed order (prepare and exact make the same)."""
    g = _gen(seed)
    s = SimpleNamespace(case=case)
    f = case["family"]
    if f == "linear":
        s.w = _linear_parts(g, case)
        s.x = _randn(g, case["rows"], s.w[5], dt=_fmt(case)[0])
    elif f == "moe":
        s.p = _moe_parts(g, case)
        s.x = _popular(g, s.p, case["skew"], case["rows"], _fmt(case)[0])
    elif f == "stack":
        s.x = _randn(g, 1, H, dt=_fmt(case)[0])
        s.layers = [_moe_parts(g, case) for _ in range(case["layers"])]
    elif f == "decoder":
        s.x = _randn(g, 1, H, dt=torch.bfloat16)
        s.layers = _decoder_parts(g, case)
    elif f == "talker":
        s.p = _talker_parts(g, torch.bfloat16)
        s.x = _randn(g, case["rows"], TH, dt=torch.bfloat16)
    else:
        s.x = _randn(g, 1, TH, dt=torch.bfloat16)
        s.layers = [_talker_parts(g, torch.bfloat16, 0.5) for _ in range(case["layers"])]
    return s


def prepare(case, seed):
    pkg = _package()
    s = _make(case, seed)
    st = SimpleNamespace(case=case, x=s.x)
    f = case["family"]
    if f == "linear":
        packed, scale, zeros, group, n, k = s.w
        w = _q(s.w) if case["fmt"] == "ct" else pkg.QWeight.awq(packed, scale, zeros, group)
        st.lin = pkg.PackedLinear.from_qweight(w, repack=case["fmt"] == "ct")
    elif f == "moe":
        st.moe = _moe_module(s.p)
    elif f == "stack":
        st.layers = [_moe_module(p).stack_entry() for p in s.layers]
        st.ws = pkg.Workspace()
    elif f == "decoder":
        layers = []
        for p in s.layers:
            qkv = pkg.PackedQKV.from_qweights(_q(p.wq), _q(p.wk), _q(p.wv))
            attn = pkg.ThinkerAttention(qkv, pkg.PackedLinear.from_qweight(_q(p.wo)), p.qn, p.kn,
                                        p.inn, NH, NKV, HD, EPS, THETA, max_len=4096)
            attn.k_cache[:, :case["pos"]].copy_(p.k)
            attn.v_cache[:, :case["pos"]].copy_(p.v)
            p.k = p.v = None
            layers.append(pkg.ThinkerDecoderLayer(attn, _moe_module(p)))
        st.dec = pkg.ThinkerDecoder(layers)
        # the rows that a step appends to the caches are part of its result
        st.rows = [c[:, case["pos"]] for l in layers for c in (l.attn.k_cache, l.attn.v_cache)]
    elif f == "talker":
        st.moe = _talker_module(s.p, case["q8"])
    else:
        mods = [_talker_module(p, case["q8"]) for p in s.layers]
        st.token = s.x.clone()

        def chain():
            h = st.token
            for m in mods:
                h = m(h, residual=h)
            return h

        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            chain()
        torch.cuda.current_stream().wait_stream(side)
        st.mods, st.graph = mods, torch.cuda.CUDAGraph()
        with torch.cuda.graph(st.graph):
            st.out = chain()
    return st


def run(state):
    f = state.case["family"]
    if f == "linear":
        return state.lin(state.x)
    if f in ("moe", "talker"):
        return state.moe(state.x, residual=state.x)
    if f == "stack":
        return _package().moe_stack(state.x, state.layers, TOPK, workspace=state.ws)
    if f == "decoder":
        return [state.dec.step(state.x, state.case["pos"]), *state.rows]
    state.token.copy_(state.x)
    state.graph.replay()
    return state.out


# ---------------------------------------------------------------------------- the measure
def _packed_bytes(case, n, k):
    """Bytes of one [n, k] int4 matrix with its scales and zero points."""
    _, group, zp = _fmt(case)
    return n * k / 2 + n * (k // group) * 2 + (n * -(-(k // group) // 8) * 4 if zp else 0)


def _hit(experts, k, rows):
    """Experts that rows tokens of top-k reach, evenly routed."""
    return experts * (1.0 - (1.0 - k / experts) ** rows)


def _moe_work(case, rows):
    per = _packed_bytes(case, 2 * I, H) + _packed_bytes(case, H, I)
    return (_hit(E, TOPK, rows) * per + E * H * 2 + H * 2 + 2 * rows * H * 2,
            2.0 * rows * (TOPK * 3 * H * I + E * H))


def _talker_work(q8, rows):
    per = 3 * TI * TH * (1 if q8 else 2) + ((2 * TI + TH) * 2 if q8 else 0)
    return (_hit(TE, TK, rows) * per + 3 * TIS * TH * 2 + TE * TH * 2 + TH * 2
            + 2 * rows * TH * 2, 2.0 * rows * (3 * TH * (TK * TI + TIS) + TE * TH))


def work(case):
    f = case["family"]
    if f == "linear":
        k, n = SHAPES[case["shape"]]
        b, fl = _packed_bytes(case, n, k) + case["rows"] * (n + k) * 2, 2.0 * case["rows"] * n * k
    elif f == "moe":
        b, fl = _moe_work(case, case["rows"])
    elif f == "stack":
        b, fl = (v * case["layers"] for v in _moe_work(case, 1))
    elif f == "decoder":
        mb, mf = _moe_work(case, 1)
        n = (NH + 2 * NKV) * HD
        ab = (_packed_bytes(case, n, H) + _packed_bytes(case, H, NH * HD)
              + 2 * NKV * HD * (case["pos"] + 1) * 2)
        af = 2.0 * (n * H + H * NH * HD) + 4.0 * NH * HD * (case["pos"] + 1)
        b, fl = (mb + ab) * case["layers"], (mf + af) * case["layers"]
    elif f == "talker":
        b, fl = _talker_work(case["q8"], case["rows"])
    else:
        b, fl = (v * case["layers"] for v in _talker_work(case["q8"], 1))
    return {"bytes": b, "flops": fl}


def tolerance(case):
    """About four times the error against 64 bits: one rounding of the result for a single
    layer (fp16 2.2e-4, bf16 1.9e-3); in the chains of layers a rounding in one travels
    through all that follow, and now and then changes an expert."""
    if case["family"] in ("decoder", "chain"):
        return {"rel": 3e-2}
    if case["family"] == "stack":
        return {"rel": 2e-2}
    fp16 = case["family"] != "talker" and case["fmt"] == "awq"
    return {"rel": 1e-3 if fp16 else 8e-3}


# ------------------------------------------------------------------------- 64-bit results
def _nibbles(words):
    """[..., m] int32 words -> [..., 8 m] float64 nibbles, low nibble first."""
    sh = torch.arange(0, 32, 4, device=words.device, dtype=torch.int32)
    return ((words.unsqueeze(-1) >> sh) & 15).flatten(-2).double()


def _dense(w, e=0):
    """Expert e of CT rows in float64."""
    packed, scale, zeros, group, n, k = w
    q = _nibbles(packed[e])
    z = 8.0 if zeros is None else _nibbles(zeros[e])[:, :k // group].repeat_interleave(group, 1)
    return (q - z) * scale[e].double().repeat_interleave(group, 1)


def _dense_awq(w):
    """AutoAWQ words in float64 as [n, k]."""
    packed, scale, zeros, group, n, k = w
    slot = torch.tensor([0, 4, 1, 5, 2, 6, 3, 7], device=DEV)  # nibble of column 8 m + i

    def cols(t):
        return _nibbles(t).view(t.shape[0], -1, 8)[..., slot].reshape(t.shape[0], -1)

    z = cols(zeros[0]).repeat_interleave(group, 0)
    return ((cols(packed[0]) - z) * scale[0].double().repeat_interleave(group, 0)).t()


def _norm(x, w, dt):
    """RMSNorm in float64, rounded to the activation type as the decoder's norm returns it."""
    y = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)
    return (y.to(dt).double() * w.double()).to(dt).double()


def _silu(v):
    return v * torch.sigmoid(v)


def _route(xn, rw, k, dt):
    """Selected experts and weights; logits round to the activation type (they decide), and
    equal ones go to the lower expert."""
    lg = (xn @ rw.double().t()).to(dt).double()
    order = torch.sort(lg, dim=-1, descending=True, stable=True).indices[:, :k]
    w = torch.softmax(lg, -1).gather(1, order)
    return order, w / w.sum(-1, keepdim=True)


def _experts(xn, sel, wts, gate_up, down, out):
    """out + the routing-weighted experts; gate_up(e) and down(e) are float64 matrices."""
    for e in torch.unique(sel).tolist():
        t, j = torch.nonzero(sel == e, as_tuple=True)
        gu = xn[t] @ gate_up(e).t()
        i = gu.shape[1] // 2
        y = (_silu(gu[:, :i]) * gu[:, i:]) @ down(e).t()
        out.index_add_(0, t, y * wts[t, j].unsqueeze(1))
    return out


def _moe_exact(h, p, dt):
    xn = _norm(h, p.nw, dt)
    sel, wts = _route(xn, p.rw, TOPK, dt)
    return _experts(xn, sel, wts, lambda e: _dense(p.gu, e), lambda e: _dense(p.dn, e), h.clone())


def _q8(w):
    """Per-output-row symmetric int8 in the weights' type, as float64 values."""
    s = w.abs().amax(dim=-1, keepdim=True).clamp_min(1e-8) / 127.0
    return (w / s).round().clamp(-127, 127).double() * s.double()


def _talker_exact(h, p, q8):
    dt = torch.bfloat16
    sel, wts = _route(h, p.rw, TK, dt)
    mat = _q8 if q8 else lambda w: w.double()
    gu = h @ p.sgu.double().t()
    shared = (_silu(gu[:, :TIS]) * gu[:, TIS:]) @ p.sdn.double().t()
    gate = torch.sigmoid(h @ p.sgw.double()).unsqueeze(1)
    return _experts(h, sel, wts, lambda e: mat(p.gu[e]), lambda e: mat(p.dn[e]),
                    h + gate * shared)


def _rotary(x, pos):
    f = _inv_freq().to(DEV).double() * pos
    f = torch.cat([f, f])
    half = torch.cat([-x[..., HD // 2:], x[..., :HD // 2]], -1)
    return x * f.cos() + half * f.sin()


def _attention_exact(h, p, pos):
    dt = torch.bfloat16
    xn = _norm(h, p.inn, dt)

    def head_norm(x, w):
        return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()

    q = _rotary(head_norm((xn @ _dense(p.wq).t()).view(NH, HD), p.qn), pos)
    k = _rotary(head_norm((xn @ _dense(p.wk).t()).view(NKV, HD), p.kn), pos)
    v = (xn @ _dense(p.wv).t()).view(NKV, HD)
    keys = torch.cat([p.k.double(), k.unsqueeze(1)], 1).repeat_interleave(NH // NKV, 0)
    vals = torch.cat([p.v.double(), v.unsqueeze(1)], 1).repeat_interleave(NH // NKV, 0)
    a = torch.softmax((keys * q.unsqueeze(1)).sum(-1) / math.sqrt(HD), -1)
    o = (a.unsqueeze(-1) * vals).sum(1).reshape(1, -1)
    return h + o @ _dense(p.wo).t(), k, v


def exact(case, seed):
    s = _make(case, seed)
    h = s.x.double()
    f = case["family"]
    if f == "linear":
        return h @ (_dense(s.w) if case["fmt"] == "ct" else _dense_awq(s.w)).t()
    if f == "moe":
        return _moe_exact(h, s.p, _fmt(case)[0])
    if f == "stack":
        for p in s.layers:
            h = _moe_exact(h, p, _fmt(case)[0])
        return h
    if f == "decoder":
        rows = []
        for p in s.layers:
            h, k, v = _attention_exact(h, p, case["pos"])
            h = _moe_exact(h, p, torch.bfloat16)
            rows += [k, v]
        return [h, *rows]
    if f == "talker":
        return _talker_exact(h, s.p, case["q8"])
    for p in s.layers:
        h = _talker_exact(h, p, case["q8"])
    return h
