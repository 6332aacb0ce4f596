"""The workloads this framework's speed is measured on.

Each listed case is work a program has the framework do through its public entry points:
one MoE decode layer, a decode stack, whole MoE blocks of the Qwen and the DeepSeek form from
one token to a long prompt, the pre-MoE norm and router, an MTP verify step with its LM head.
Shapes are the repository's own configurations: the benchmark's (hidden 2048 / intermediate
512 / 512 experts / top 10; 7168 / 2048 / 256 / top 8 in 8 groups) and the reference models'
(2560 / 640 / 512 / top 10; 5120 / 2304 / 384 / top 6).

``draw`` spreads the same kinds of work over the token counts, shapes, layouts and formats
the listed cases stand for. ``exact`` restates each case in 64-bit torch.
"""
from __future__ import annotations

import math
from dataclasses import replace
from types import SimpleNamespace

import torch

import whallm_amd as wa
from whallm_amd import operators as O
from whallm_amd import synthetic as S
from whallm_amd.ops import DecodeLayer, PersistentDecodeStack
from whallm_amd.verify import VerifyStep

# hidden, intermediate, experts, top k
QWEN = {"2048": (2048, 512, 512, 10), "2560": (2560, 640, 512, 10), "4096": (4096, 2048, 128, 8)}
# form: hidden, intermediate, experts, top k, groups, kept groups, score function, SwiGLU limit
DEEPSEEK = {
    "fp8-128": (7168, 2048, 256, 8, 8, 4, "sigmoid", 0.0),       # fp32 128 x 128 block scales
    "fp8-32": (5120, 2304, 384, 6, 1, 1, "sqrtsoftplus", 10.0),  # E8M0 32 x 32 block scales
    "mxfp4": (5120, 2304, 384, 6, 1, 1, "sqrtsoftplus", 10.0),   # routed and shared experts in MXFP4
}
ROUTE_SCALE = 2.5
VOCAB = 129280
EPS = 1e-6


# ------------------------------------------------------------------------------- the cases

def listed():
    return [
        # a runtime that calls its MoE half once per decoder layer, between attention blocks
        {"name": "layer-decode", "kind": "layer", "hidden": 2048, "experts": 512, "k": 10},
        # one token through a resident stack (the decode benchmark's layers, 8 of them)
        {"name": "stack-decode", "kind": "stack", "layers": 8, "experts": 512, "k": 10},
        # the Qwen block as its operator runs it (router, routed experts, bf16 shared expert):
        # one decode token; the 8 rows of a speculative verify round; a short ragged prompt; a
        # prompt chunk on weights repacked once for prefill
        {"name": "qwen-decode-1", "kind": "qwen", "shape": "2560", "tokens": 1, "tiled": False},
        {"name": "qwen-verify-8", "kind": "qwen", "shape": "2560", "tokens": 8, "tiled": False},
        {"name": "qwen-prompt-301", "kind": "qwen", "shape": "2048", "tokens": 301, "tiled": False},
        {"name": "qwen-prompt-2048", "kind": "qwen", "shape": "2560", "tokens": 2048, "tiled": True},
        # a 16K-token prefill of one MXFP4 layer with skewed routing and an MXFP4 shared expert
        {"name": "mxfp4-prefill-16384", "kind": "mxfp4", "tokens": 16384, "terms": "e4m3"},
        # the DeepSeek block (scored router, routed and shared experts): one decode token and a
        # 4096-token prefill in FP8, a small batch of decode requests in MXFP4
        {"name": "deepseek-decode-1", "kind": "deepseek", "form": "fp8-128", "tokens": 1, "tiled": False},
        {"name": "deepseek-batch-64", "kind": "deepseek", "form": "mxfp4", "tokens": 64, "tiled": False},
        {"name": "deepseek-prefill-4096", "kind": "deepseek", "form": "fp8-128", "tokens": 4096, "tiled": True},
        # an accepted token and three drafts through FP8 layers, the LM head and acceptance
        {"name": "verify-4", "kind": "verify", "layers": 2, "rows": 4},
        # the residual add, norm, router and top-k before a prompt's MoE
        {"name": "router-prompt-4000", "kind": "router", "shape": "2560", "tokens": 4000},
    ]


def _tokens(rng, low, high):
    return max(low, min(high, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["layer", "stack", "qwen", "qwen", "qwen", "mxfp4", "deepseek", "deepseek", "deepseek", "verify",
                       "router"])
    if kind == "layer":
        return {"kind": kind, "hidden": rng.choice([1024, 2048]), "experts": rng.randint(32, 512), "k": rng.randint(2, 11)}
    if kind == "stack":
        return {"kind": kind, "layers": rng.randint(2, 10), "experts": 8 * rng.randint(4, 64), "k": rng.randint(2, 11)}
    if kind == "qwen":
        t = _tokens(rng, 1, 4096)
        return {"kind": kind, "shape": rng.choice(sorted(QWEN)), "tokens": t, "tiled": t >= 512 and rng.random() < 0.5}
    if kind == "mxfp4":
        return {"kind": kind, "tokens": _tokens(rng, 512, 16384), "terms": rng.choice(["e4m3", "e4m3", "e2m3"])}
    if kind == "deepseek":
        t = _tokens(rng, 1, 3000)
        return {"kind": kind, "form": rng.choice(sorted(DEEPSEEK)), "tokens": t, "tiled": t >= 512 and rng.random() < 0.5}
    if kind == "verify":
        return {"kind": kind, "layers": rng.randint(1, 3), "rows": rng.randint(2, 8)}
    return {"kind": kind, "shape": rng.choice(["2048", "2560", "deepseek"]), "tokens": _tokens(rng, 1, 16384)}


# ------------------------------------------------------------------------------- inputs

class _Layer:
    """The cache interface of a program whose experts are all resident: one table for the layer."""

    def __init__(self, table):
        self.table = table

    def current_batched(self, layer):
        return self.table


def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _bf16(g, *shape, std=1.0):
    return (torch.randn(*shape, device="cuda", generator=g) * std).to(torch.bfloat16)


def _mxfp4(g, experts, hidden, inter, **kw):
    t = S.mxfp4_experts_device(experts, hidden, inter, "cuda", g)
    t.gate_up_scales.sub_(4)  # projections of N(0, 1) inputs of order one
    t.down_scales.sub_(2)
    return replace(t, **kw)


def _fp8(g, experts, hidden, inter, fmt):
    return S.fp8_experts_device(experts, hidden, inter, "cuda", g, scale_format=fmt)


def _router_shape(shape):
    """hidden, experts, k, whether the layer has a shared gate (the Qwen form)."""
    if shape == "deepseek":
        H, _, E, k = DEEPSEEK["fp8-128"][:4]
        return H, E, k, False
    H, _, E, k = QWEN[shape]
    return H, E, k, True


def _inputs(case, seed):
    """Everything of a case in the row layout: tables, vectors, tokens."""
    g, kind = _gen(seed), case["kind"]
    s = SimpleNamespace()
    if kind == "layer":
        H, E = case["hidden"], case["experts"]
        s.experts, s.shared = _mxfp4(g, E, H, 512), _mxfp4(g, 1, H, 512)
        s.router = _bf16(g, E, H, std=H ** -0.5)
        s.gate = _bf16(g, H, std=0.02)
        s.norm = (1 + torch.randn(H, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
        s.residual = torch.randn(H, device="cuda", generator=g)
    elif kind == "stack":
        H, E, L = 2048, case["experts"], case["layers"]
        s.layers = [_mxfp4(g, E, H, 512) for _ in range(L)]
        s.shared = [_mxfp4(g, 1, H, 512) for _ in range(L)]
        s.gates = [_bf16(g, H, std=0.02) for _ in range(L)]
        s.logits = torch.randn(L, E, device="cuda", generator=g)
        s.residual = torch.randn(H, device="cuda", generator=g)
    elif kind == "qwen":
        H, I, E, k = QWEN[case["shape"]]
        s.experts = _mxfp4(g, E, H, I)
        s.router, s.gate = _bf16(g, E, H, std=H ** -0.5), _bf16(g, 1, H, std=0.02)
        s.w1, s.w3, s.w2 = _bf16(g, I, H, std=H ** -0.5), _bf16(g, I, H, std=H ** -0.5), _bf16(g, H, I, std=I ** -0.5)
        s.x = _bf16(g, 1, case["tokens"], H)
    elif kind == "mxfp4":
        H, I, E, k = QWEN["2048"]
        s.experts, s.shared = _mxfp4(g, E, H, I), _mxfp4(g, 1, H, I)
        s.gate = _bf16(g, H, std=0.02)
        skew = torch.from_numpy(S.zipf_bias(E, 1.1)).to("cuda")[torch.randperm(E, device="cuda", generator=g)]
        s.logits = torch.randn(case["tokens"], E, device="cuda", generator=g) + skew
        s.x = _bf16(g, case["tokens"], H)
    elif kind == "deepseek":
        H, I, E, k, _, _, _, _ = DEEPSEEK[case["form"]]
        if case["form"] == "mxfp4":
            s.experts, s.shared = _mxfp4(g, E, H, I, up_first=True), _mxfp4(g, 1, H, I, up_first=True)
        else:
            fmt = 1 if case["form"] == "fp8-32" else 0
            s.experts, s.shared = _fp8(g, E, H, I, fmt), _fp8(g, 1, H, I, fmt)
        s.router = _bf16(g, E, H, std=H ** -0.5)
        s.bias = torch.randn(E, device="cuda", generator=g) * 0.1
        s.x = _bf16(g, 1, case["tokens"], H)
    elif kind == "verify":
        H, I, E, k = DEEPSEEK["fp8-128"][:4]
        L, M = case["layers"], case["rows"]
        s.layers = [_fp8(g, E, H, I, 0) for _ in range(L)]
        s.shared = [_fp8(g, 1, H, I, 0) for _ in range(L)]
        s.biases = [torch.randn(E, device="cuda", generator=g) * 0.1 for _ in range(L)]
        # LM-head rows of uneven norm, so a row's largest logit stands clear as a model's does
        norm = torch.exp(torch.randn(VOCAB, 1, device="cuda", generator=g) * 0.7)
        s.head = (torch.randn(VOCAB, H, device="cuda", generator=g) * norm * H ** -0.5).to(torch.bfloat16)
        s.logits = torch.randn(L, M, E, device="cuda", generator=g)
        s.residual = torch.randn(M, H, device="cuda", generator=g)
        s.drafts = torch.randint(0, VOCAB, (M - 1,), device="cuda", generator=g, dtype=torch.int32)
    else:
        H, E, k, gated = _router_shape(case["shape"])
        s.router = _bf16(g, E, H, std=H ** -0.5)
        s.gate = _bf16(g, H, std=0.02) if gated else None
        s.norm = (1 + torch.randn(H, device="cuda", generator=g) * 0.1).to(torch.bfloat16)
        s.bias = None if gated else torch.randn(E, device="cuda", generator=g) * 0.1
        s.residual = torch.randn(case["tokens"], H, device="cuda", generator=g)
        s.y = _bf16(g, case["tokens"], H, std=0.5)
    return s


def prepare(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    s.case = case
    if kind == "layer":
        s.call = DecodeLayer(s.experts, s.router, s.shared, s.gate, k=case["k"], norm_weight=s.norm, eps=EPS)
        s.out = torch.empty_like(s.residual)
        s.y = torch.empty(case["hidden"], dtype=torch.bfloat16, device="cuda")
    elif kind == "stack":
        s.call = PersistentDecodeStack(s.layers, s.shared, s.gates, k=case["k"], eps=EPS)
        s.x_out = torch.empty(2048, dtype=torch.bfloat16, device="cuda")
    elif kind == "qwen":
        H, I, E, k = QWEN[case["shape"]]
        table = wa.prefill_layout(s.experts) if case["tiled"] else s.experts
        args = SimpleNamespace(hidden_size=H, num_experts=E, shared_expert_intermediate_size=I, num_experts_per_tok=k,
                               norm_topk_prob=True)
        s.call = O.SparseMoE(args, 0, _Layer(table))
        s.call.gate.weight, s.call.shared_expert_gate.weight = s.router, s.gate
        mlp = s.call.shared_expert
        mlp.gate_proj.weight, mlp.up_proj.weight, mlp.down_proj.weight = s.w1, s.w3, s.w2
        s.experts = table
    elif kind == "mxfp4":
        s.experts = replace(wa.prefill_layout(s.experts), act_terms=case["terms"])
        s.shared = replace(wa.prefill_layout(s.shared), act_terms=case["terms"])
    elif kind == "deepseek":
        H, I, E, k, groups, kept, func, limit = DEEPSEEK[case["form"]]
        if case["tiled"]:
            s.experts, s.shared = wa.prefill_layout(s.experts), wa.prefill_layout(s.shared)
        s.gate = O.Gate(H, E, k, func, ROUTE_SCALE, True, 1.0, groups, kept)
        s.gate.weight, s.gate.bias = s.router, s.bias
        s.call = O._StreamingSwitchGLU(0, _Layer(s.experts), O.ClampedSwiGLU(limit) if limit else O.SwiGLU())
    elif kind == "verify":
        s.call = VerifyStep(s.layers, s.shared, s.biases, s.head, k=8, route_scale=ROUTE_SCALE, eps=EPS)
    else:
        s.packed = wa.repack_router(s.router, s.gate)
        s.v = torch.empty_like(s.residual)
    return s


def run(s):
    kind = s.case["kind"]
    if kind == "layer":
        return {"residual": s.call(s.residual, s.out, s.y), "y": s.y}
    if kind == "stack":
        # the stack updates the residual stream in place: a token starts from its own copy
        r = s.call(s.logits, s.residual.clone(), s.x_out, check=False)
        return {"residual": r, "x": s.x_out}
    if kind == "qwen":
        return s.call(s.x)
    if kind == "mxfp4":
        idx, w = wa.route_softmax_topk(s.logits, 10)
        return wa.moe_mxfp4(s.x, idx, w, s.experts, s.shared, s.gate)
    if kind == "deepseek":
        return O.streaming_moe(s.gate, s.call, s.shared, s.x)
    if kind == "verify":
        r = s.residual.clone()
        acceptance, logits = s.call(s.logits, r, s.drafts)
        return {"logits": logits, "residual": r, "acceptance": acceptance}
    x, logits, shared = wa.norm_router(s.residual, s.y, s.router, s.gate, s.norm, EPS, s.v, s.packed)
    if s.gate is not None:
        idx, w = wa.route_softmax_topk(logits, 10)
    else:
        idx, w = wa.route_scored(logits, s.bias, 8, "sigmoid", ROUTE_SCALE, True, 8, 4)
    return {"x": x, "logits": logits, "shared": shared, "v": s.v, "idx": idx, "w": w}


# ------------------------------------------------------------------------------- work

def _touched(experts, k, tokens):
    """Experts that `tokens` tokens of k uniform choices each reach, on average."""
    return experts * (1 - (1 - k / experts) ** tokens)


def _mx_bytes(H, I):
    return 3 * H * I // 2 + 3 * H * I // 32


def _fp8_bytes(H, I, form):
    return 3 * H * I + (3 * H * I // 1024 if form == "fp8-32" else 3 * H * I // 16384 * 4)


def work(case):
    kind = case["kind"]
    if kind == "layer":
        H, E, k = case["hidden"], case["experts"], case["k"]
        return {"bytes": (k + 1) * _mx_bytes(H, 512) + E * H * 2 + H * (4 + 4 + 2 + 2 + 2),
                "flops": 2 * H * (3 * 512 * (k + 1) + E)}
    if kind == "stack":
        L, E, k = case["layers"], case["experts"], case["k"]
        return {"bytes": L * ((k + 1) * _mx_bytes(2048, 512) + E * 4 + 4096) + 2048 * 10,
                "flops": L * 2 * 2048 * 3 * 512 * (k + 1)}
    if kind == "qwen":
        H, I, E, k = QWEN[case["shape"]]
        T = case["tokens"]
        return {"bytes": _touched(E, k, T) * _mx_bytes(H, I) + 2 * (E * H + 3 * H * I + H) + 4 * T * H,
                "flops": 2 * T * H * (3 * I * (k + 1) + E)}
    if kind == "mxfp4":
        H, I, E, k = QWEN["2048"]
        T = case["tokens"]
        return {"bytes": (_touched(E, k, T) + 1) * _mx_bytes(H, I) + 4 * T * (H + E), "flops": 2 * T * H * 3 * I * (k + 1)}
    if kind == "deepseek":
        H, I, E, k = DEEPSEEK[case["form"]][:4]
        T = case["tokens"]
        per = _mx_bytes(H, I) if case["form"] == "mxfp4" else _fp8_bytes(H, I, case["form"])
        return {"bytes": (_touched(E, k, T) + 1) * per + 2 * E * H + 4 * T * H,
                "flops": 2 * T * H * (3 * I * (k + 1) + E)}
    if kind == "verify":
        H, I, E, k = DEEPSEEK["fp8-128"][:4]
        L, M = case["layers"], case["rows"]
        return {"bytes": L * (_touched(E, k, M) + 1) * _fp8_bytes(H, I, "fp8-128") + VOCAB * (2 * H + 4 * M),
                "flops": 2 * M * H * (L * 3 * I * (k + 1) + VOCAB)}
    H, E, k, gated = _router_shape(case["shape"])
    T = case["tokens"]
    return {"bytes": T * H * (4 + 2 + 2 + 4) + T * E * 4 + 2 * E * H + T * k * 8, "flops": 2 * T * H * (E + 1)}


def tolerance(case):
    """About four times each path's distance from its 64-bit restatement."""
    kind = case["kind"]
    if kind == "router":
        # fp32 sums of bf16 products; a value of x on a rounding boundary moves by one bf16 step
        return {"rel": 1e-4, "max": 2e-2, "differ": 1e-3}
    if kind == "layer":
        return {"rel": 7e-3, "max": 0.1}
    if kind in ("stack", "verify"):  # rounding travels through the layers
        return {"rel": 2e-2, "max": 0.3}
    return {"rel": 1e-2, "max": 0.3}


# ------------------------------------------------------------------------------- 64 bits

_E2M1 = (0.0, 0.5, 1.0, 1.5, 2.0, 3.0, 4.0, 6.0, -0.0, -0.5, -1.0, -1.5, -2.0, -3.0, -4.0, -6.0)


def _dequant_mx(words, scales):
    b = words.view(torch.uint8)
    lut = torch.tensor(_E2M1, dtype=torch.float64, device=words.device)
    v = torch.stack([lut[(b & 15).long()], lut[(b >> 4).long()]], dim=-1).reshape(words.shape[0], -1)
    return v * torch.exp2(scales.double() - 127).repeat_interleave(32, dim=1)


def _dequant_f8(codes, scales):
    n = 32 if scales.dtype == torch.uint8 else 128
    s = torch.exp2(scales.double() - 127) if n == 32 else scales.double()
    return codes.view(torch.float8_e4m3fn).to(torch.float32).double() * s.repeat_interleave(n, 0).repeat_interleave(n, 1)


def _ffn(x, table, e, limit=0.0):
    if hasattr(table, "w13"):
        w13, w2 = _dequant_f8(table.w13[e], table.w13_scales[e]), _dequant_f8(table.w2[e], table.w2_scales[e])
    else:
        w13, w2 = _dequant_mx(table.gate_up[e], table.gate_up_scales[e]), _dequant_mx(table.down[e], table.down_scales[e])
    a, b = (x @ w13.T).chunk(2, dim=1)
    g, u = (b, a) if table.up_first else (a, b)
    if limit:
        g, u = g.clamp(max=limit), u.clamp(-limit, limit)
    return (torch.nn.functional.silu(g) * u) @ w2.T


def _experts(x, idx, w, table, limit=0.0):
    y = torch.zeros_like(x)
    flat, order = idx.reshape(-1).sort()
    ids, counts = torch.unique_consecutive(flat, return_counts=True)
    at = 0
    for e, n in zip(ids.tolist(), counts.tolist()):
        pair = order[at:at + n]
        at += n
        t = pair // idx.shape[1]
        y.index_add_(0, t, _ffn(x[t], table, e, limit) * w.reshape(-1)[pair, None])
    return y


def _softmax_topk(logits, k):
    v, i = logits.topk(k, dim=-1)
    return i, torch.softmax(v, dim=-1)


def _scored_topk(logits, bias, k, func, groups, kept):
    s = torch.sigmoid(logits) if func == "sigmoid" else torch.nn.functional.softplus(logits).sqrt()
    b = s + bias.double()
    if groups > 1:
        top = b.reshape(len(b), groups, -1).topk(2, dim=-1)[0].sum(-1).topk(kept, dim=-1)[1]
        keep = torch.zeros(len(b), groups, dtype=torch.bool, device=b.device).scatter_(1, top, True)
        b = b.masked_fill(~keep.repeat_interleave(b.shape[1] // groups, dim=1), -math.inf)
    i = b.topk(k, dim=-1)[1]
    w = s.gather(1, i)
    return i, w / w.sum(-1, keepdim=True) * ROUTE_SCALE


def _norm(v, weight=None):
    x = v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS)
    x = x if weight is None else x * weight.double()
    return x.to(torch.bfloat16).double()  # the entry points hand x on as bf16


def exact(case, seed):
    s, kind = _inputs(case, seed), case["kind"]
    if kind == "layer":
        r = s.residual.double()[None]
        x = _norm(r, s.norm)
        idx, w = _softmax_topk(x @ s.router.double().T, case["k"])
        y = _experts(x, idx, w, s.experts) + torch.sigmoid(x @ s.gate.double())[:, None] * _ffn(x, s.shared, 0)
        return {"residual": (r + y)[0], "y": y[0]}
    if kind == "stack":
        r = s.residual.double()[None]
        for l, (table, sh) in enumerate(zip(s.layers, s.shared)):
            x = _norm(r)
            idx, w = _softmax_topk(s.logits[l:l + 1].double(), case["k"])
            r = r + _experts(x, idx, w, table) + torch.sigmoid(x @ s.gates[l].double())[:, None] * _ffn(x, sh, 0)
        return {"residual": r[0], "x": _norm(r)[0]}
    if kind == "qwen":
        k, x = QWEN[case["shape"]][3], s.x[0].double()
        idx, w = _softmax_topk(x @ s.router.double().T, k)
        mlp = (torch.nn.functional.silu(x @ s.w1.double().T) * (x @ s.w3.double().T)) @ s.w2.double().T
        return (_experts(x, idx, w, s.experts) + torch.sigmoid(x @ s.gate.double().T) * mlp)[None]
    if kind == "mxfp4":
        x = s.x.double()
        idx, w = _softmax_topk(s.logits.double(), 10)
        return _experts(x, idx, w, s.experts) + torch.sigmoid(x @ s.gate.double())[:, None] * _ffn(x, s.shared, 0)
    if kind == "deepseek":
        H, I, E, k, groups, kept, func, limit = DEEPSEEK[case["form"]]
        x = s.x[0].double()
        idx, w = _scored_topk(x @ s.router.double().T, s.bias, k, func, groups, kept)
        return (_experts(x, idx, w, s.experts, limit) + _ffn(x, s.shared, 0, limit))[None]
    if kind == "verify":
        r = s.residual.double()
        for l, (table, sh) in enumerate(zip(s.layers, s.shared)):
            x = _norm(r)
            idx, w = _scored_topk(s.logits[l].double(), s.biases[l], 8, "sigmoid", 8, 4)
            r = r + _experts(x, idx, w, table) + _ffn(x, sh, 0)
        x = _norm(r)
        logits = torch.cat([x @ h.double().T for h in s.head.split(16384)], dim=1)
        return {"logits": logits, "residual": r, "acceptance": None}
    v = s.residual.double() + s.y.double()
    x = _norm(v, s.norm)
    logits = x @ s.router.double().T
    if s.gate is not None:
        idx, w = _softmax_topk(logits, 10)
        shared = x @ s.gate.double()
    else:
        idx, w = _scored_topk(logits, s.bias, 8, "sigmoid", 8, 4)
        shared = None
    return {"x": x, "logits": logits, "shared": shared, "v": v, "idx": None, "w": w}
