"""The work a program has this package do, as cases that can be timed and checked.

Every case is one layer or block, called as a serving program (or the store writer) calls
it, through the package's public functions.  The kinds:

* ``linear``  -- one int8 qrow linear in the store's fp32 (or a 16-bit) compute dtype;
* ``layer``   -- the int8 linears of one bf16 decoder layer: q/k/v in one call, the output
  projection, the paired gate/up SwiGLU and the down projection.  Attention and norms run
  elsewhere, so their results (the inputs of o and of the MLP) are inputs here;
* ``head``    -- the fused top-2 search over a vocabulary head and its fp32 rerank;
* ``w8a8``    -- the W8A8 linear, activations quantized per token, outlier columns protected;
* ``moe``     -- router, route and int8 experts of one routed layer;
* ``lowbit``  -- a packed int3 / int2 linear;
* ``encode``  -- the store writer's codecs on fp32 weights.

``listed()`` holds one to three sizes of each, ``draw`` any size of the same ranges.
"""

from __future__ import annotations

import math

import torch

import __graft_entry__

__graft_entry__.load_package()

from mrun_pub_amd import codecs, lowbit, moe, qrow, w8a8  # noqa: E402

DEV = "cuda:0"
_DT = {"f32": torch.float32, "bf16": torch.bfloat16, "f16": torch.float16}

# The largest amounts of work of each kind; draws stay below them.
MAX_LAYER_MACS = 1531 * (1536 * (1536 + 2 * 256) + 1536 * 1536 + 3 * 1536 * 8960)
MAX_LINEAR_MACS = 149 * 1536 * 8960
MAX_LOWBIT_MACS = 131 * 4096 * 11008
MAX_W8A8_MACS = 2048 * 14336 * 4096


def listed() -> list[dict]:
    return [
        # A projection of a small fp32 store, one token: the smallest call there is.
        {"name": "linear_f32_m1", "kind": "linear", "m": 1, "n": 4096, "k": 1024, "dtype": "f32", "row_stable": False},
        # The same store taking in a prompt: the fp32 down projection for 149 tokens.
        {"name": "linear_f32_m149", "kind": "linear", "m": 149, "n": 1536, "k": 8960, "dtype": "f32",
         "row_stable": False},
        # Decode of one sequence, a whole layer's linears.
        {"name": "layer_m1", "kind": "layer", "m": 1, "hidden": 1536, "kv": 256, "inter": 8960},
        # Decode of a batch that is not a round number.
        {"name": "layer_m23", "kind": "layer", "m": 23, "hidden": 1536, "kv": 256, "inter": 8960},
        # Prefill of a prompt.
        {"name": "layer_m1531", "kind": "layer", "m": 1531, "hidden": 1536, "kv": 256, "inter": 8960},
        # Greedy decoding of a batch: the next tokens from the vocabulary head.
        {"name": "head_m11", "kind": "head", "m": 11, "vocab": 151936, "rows": 151665, "k": 1536, "dtype": "bf16"},
        # W8A8 prefill with eight protected columns.
        {"name": "w8a8_m2048", "kind": "w8a8", "m": 2048, "n": 14336, "k": 4096, "protect": 8, "out": "bf16"},
        # Routed experts in decode of a small batch, weight-only math.
        {"name": "moe_t13", "kind": "moe", "t": 13, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768,
         "w8a16": True},
        # Routed experts in prefill, W8A8 math.
        {"name": "moe_t777", "kind": "moe", "t": 777, "experts": 128, "top_k": 8, "hidden": 2048, "inter": 768,
         "w8a16": False},
        # One token through a group-of-64 int3 linear with zero points.
        {"name": "int3_m1", "kind": "lowbit", "bits": 3, "m": 1, "n": 11008, "k": 4096, "group": 64, "dtype": "bf16"},
        # A short prompt through an int2 linear of the writers' own layout.
        {"name": "int2_m131", "kind": "lowbit", "bits": 2, "m": 131, "n": 4096, "k": 11008, "group": 128,
         "dtype": "bf16"},
        # The store writer: one weight matrix to packed int3.
        {"name": "encode_int3", "kind": "encode", "bits": 3, "n": 11008, "k": 4096, "group": 128},
    ]


def _log_int(rng, lo: int, hi: int) -> int:
    """A whole number of [lo, hi], even over its logarithm, odd as often as even."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.49)))))))


def draw(rng) -> dict:
    kind = rng.choice(["linear", "layer", "layer", "head", "w8a8", "moe", "moe", "lowbit", "lowbit", "encode"])
    if kind == "linear":
        n, k = rng.choice([(4096, 1024), (1536, 8960), (2560, 1000), (8960, 1536), (rng.randrange(300, 6000), 1536),
                           (rng.randrange(300, 3000), 320)])
        dtype = rng.choice(["f32", "f32", "bf16", "f16"])
        return {"kind": kind, "m": _log_int(rng, 1, max(1, min(149, MAX_LINEAR_MACS // (n * k)))), "n": n, "k": k,
                "dtype": dtype, "row_stable": rng.random() < 0.2}
    if kind == "layer":
        hidden, kv, inter = rng.choice([(1536, 256, 8960), (1024, 512, 2816), (2048, 512, 11008), (4096, 1024, 14336)])
        macs = hidden * (2 * hidden + 2 * kv) + 3 * hidden * inter
        return {"kind": kind, "m": _log_int(rng, 1, min(1531, MAX_LAYER_MACS // macs)), "hidden": hidden, "kv": kv,
                "inter": inter}
    if kind == "head":
        vocab, rows = rng.choice([(151936, 151665), (151936, 151936), (50304, 50257), (32000, 32000)])
        return {"kind": kind, "m": _log_int(rng, 1, 11), "vocab": vocab, "rows": rows,
                "k": rng.choice([1024, 1536]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    if kind == "w8a8":
        n, k = rng.choice([(14336, 4096), (4096, 4096), (1536, 8960), (8960, 1536), (4096, 14336), (1000, 2048)])
        return {"kind": kind, "m": _log_int(rng, 8, min(2048, MAX_W8A8_MACS // (n * k))), "n": n, "k": k,
                "protect": rng.choice([0, 8, 8, 16]), "out": rng.choice(["bf16", "f32"])}
    if kind == "moe":
        experts, inter = rng.choice([(128, 768), (64, 1024)])
        return {"kind": kind, "t": _log_int(rng, 1, 777), "experts": experts, "top_k": 8, "hidden": 2048,
                "inter": inter, "w8a16": rng.random() < 0.5}
    if kind == "lowbit":
        n, k = rng.choice([(11008, 4096), (4096, 11008), (4096, 4096), (rng.randrange(301, 3000, 2), 2048)])
        return {"kind": kind, "bits": rng.choice([3, 2]), "m": _log_int(rng, 1, min(131, MAX_LOWBIT_MACS // (n * k))),
                "n": n, "k": k, "group": rng.choice([64, 128]), "dtype": rng.choice(["bf16", "bf16", "f32"])}
    n, k = rng.choice([(11008, 4096), (4096, 11008), (rng.randrange(301, 9000, 2), 1536)])
    return {"kind": "encode", "bits": rng.choice([8, 3, 2]), "n": n, "k": k, "group": 128}


# ---- inputs ------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, *shape) -> torch.Tensor:
    return torch.randn(*shape, device=DEV, generator=g)


def _qrow_weight(g, n: int, k: int) -> tuple[torch.Tensor, torch.Tensor]:
    """Row-quantized normal weights: absmax / 127 of 1/sqrt(k) rows is about 4/127 of it."""
    codes = (_randn(g, n, k) * 31.0).round_().clamp_(-127, 127).to(torch.int8)
    scales = (torch.rand(n, device=DEV, generator=g) + 0.5) / (31.0 * math.sqrt(k))
    return codes, scales


def _page(name: str, w) -> qrow.CompactQRowPage:
    return qrow.CompactQRowPage(name, 0, int(w[0].shape[0]), int(w[0].shape[1]), w[0], w[1])


def _pack(codes: torch.Tensor, bits: int) -> torch.Tensor:
    """Codes [n, k] (k % 8 == 0) to LSB-first row bitstreams."""
    n, k = codes.shape
    c = codes.view(n, k // 8, 8).to(torch.int32)
    word = torch.zeros(n, k // 8, dtype=torch.int32, device=codes.device)
    for i in range(8):
        word |= c[:, :, i] << (bits * i)
    return torch.stack([(word >> (8 * b)) & 255 for b in range(bits)], dim=2).to(torch.uint8).reshape(n, -1)


def _inputs(case: dict, seed: int) -> dict:
    g = _gen(seed)
    kind = case["kind"]
    if kind == "linear":
        return {"w": _qrow_weight(g, case["n"], case["k"]), "x": _randn(g, case["m"], case["k"]).to(_DT[case["dtype"]])}
    if kind == "layer":
        h, kv, it, m = case["hidden"], case["kv"], case["inter"], case["m"]
        shapes = {"q": (h, h), "k": (kv, h), "v": (kv, h), "o": (h, h), "gate": (it, h), "up": (it, h), "down": (h, it)}
        out = {name: _qrow_weight(g, n, k) for name, (n, k) in shapes.items()}
        for name in ("x", "attn", "mlp"):
            out[name] = _randn(g, m, h).to(torch.bfloat16)
        return out
    if kind == "head":
        return {"w": _qrow_weight(g, case["vocab"], case["k"]), "x": _randn(g, case["m"], case["k"]).to(_DT[case["dtype"]])}
    if kind == "w8a8":
        x = _randn(g, case["m"], case["k"])
        x = torch.where(torch.rand(x.shape, device=DEV, generator=g) < 0.001, x * 20.0, x)
        return {"w": _qrow_weight(g, case["n"], case["k"]), "x": x.to(torch.bfloat16)}
    if kind == "moe":
        E, H, inter, T = case["experts"], case["hidden"], case["inter"], case["t"]
        gu, gus = _qrow_weight(g, E * 2 * inter, H)
        dn, dns = _qrow_weight(g, E * H, inter)
        return {"gate_up": gu.view(E, 2 * inter, H), "gate_up_scales": gus.view(E, 2 * inter), "down": dn.view(E, H, inter),
                "down_scales": dns.view(E, H), "x": _randn(g, T, H).to(torch.bfloat16),
                "logits": _randn(g, T, E).to(torch.bfloat16)}
    if kind == "lowbit":
        n, k, bits, group = case["n"], case["k"], case["bits"], case["group"]
        # groups of 64 are the asymmetric variant (fp16 scales and zero points over the full
        # code range), groups of 128 the writers' symmetric one (fixed offset, fp32 scales)
        asym = group == 64
        ng = k // group
        lo, hi = (0, 1 << bits) if asym else ((1, 8) if bits == 3 else (0, 3))
        codes = torch.randint(lo, hi, (n, k), dtype=torch.uint8, device=DEV, generator=g)
        scales = (torch.rand(n, ng, device=DEV, generator=g) + 0.5) / math.sqrt(k)
        zeros = None
        if asym:
            scales = scales.half()
            zeros = ((1 << bits) * 0.5 + 0.5 * _randn(g, n, ng)).half()
        return {"codes": codes, "scales": scales, "zeros": zeros, "x": _randn(g, case["m"], k).to(_DT[case["dtype"]])}
    return {"w": _randn(g, case["n"], case["k"]) / math.sqrt(case["k"])}


def prepare(case: dict, seed: int) -> dict:
    d = _inputs(case, seed)
    kind = case["kind"]
    st = {"case": case}
    if kind == "linear":
        st.update(codes=d["w"][0], scales=d["w"][1], x=d["x"])
    elif kind == "layer":
        st.update({n: _page(n, d[n]) for n in ("q", "k", "v", "o", "gate", "up", "down")})
        st.update(x=d["x"], attn=d["attn"], mlp=d["mlp"])
    elif kind == "head":
        st.update(page=_page("head", d["w"]), x=d["x"])
    elif kind == "w8a8":
        st.update(codes=d["w"][0], scales=d["w"][1], x=d["x"])
    elif kind == "moe":
        layer = moe.Int8ExpertLayer.from_arrays(d["gate_up"], d["gate_up_scales"], d["down"], d["down_scales"], DEV)
        st.update(backend=moe.Int8ExpertBackend([layer], w8a16=case["w8a16"]), x=d["x"], logits=d["logits"])
    elif kind == "lowbit":
        page = lowbit.LowbitPage("w", case["bits"], case["group"], case["k"], _pack(d["codes"], case["bits"]), d["scales"],
                                 d["zeros"])
        st.update(page=page, x=d["x"])
    else:
        st.update(w=d["w"])
    return st


def run(state: dict):
    case = state["case"]
    kind = case["kind"]
    if kind == "linear":
        return qrow.qrow_matmul(state["codes"], state["scales"], state["x"], row_stable=case["row_stable"])
    if kind == "layer":
        q, k, v = qrow.qrow_matmul_multi([(state[n].codes, state[n].scales) for n in ("q", "k", "v")], state["x"])
        o, _ = qrow.fused_qrow_matmul(state["o"], state["attn"])
        act, _ = qrow.fused_qrow_swiglu(state["gate"], state["up"], state["mlp"])
        down, _ = qrow.fused_qrow_matmul(state["down"], act)
        return q, k, v, o, act, down
    if kind == "head":
        idx, val, _, _ = qrow.fused_qrow_reranked_argmax(state["page"], state["x"], semantic_row_count=case["rows"])
        return idx, val
    if kind == "w8a8":
        return w8a8.w8a8_matmul(state["codes"], state["scales"], state["x"], protect_k=case["protect"],
                                out_dtype=_DT[case["out"]])
    if kind == "moe":
        weights, experts = moe.route_topk(state["logits"], case["top_k"])
        return state["backend"].moe(0, state["x"], experts, weights), weights, experts
    if kind == "lowbit":
        return lowbit.lowbit_matmul(state["page"], state["x"])
    if case["bits"] == 8:
        return codecs.quant_row_int8(state["w"])
    fn = codecs.quant_row_int3 if case["bits"] == 3 else codecs.quant_row_int2
    return fn(state["w"], case["group"])


# ---- what a pass cannot do without ----------------------------------------------------------


def work(case: dict) -> dict:
    kind = case["kind"]
    if kind == "linear":
        m, n, k = case["m"], case["n"], case["k"]
        es = 4 if case["dtype"] == "f32" else 2
        return {"bytes": n * k + 4 * n + es * m * (n + k), "flops": 2 * m * n * k}
    if kind == "layer":
        m, h, kv, it = case["m"], case["hidden"], case["kv"], case["inter"]
        params = h * (2 * h + 2 * kv) + 3 * h * it
        rows = 2 * h + 2 * kv + 2 * it + h
        # x, attn, mlp and act in (act is also an output), q, k, v, o, act and down out
        acts = 2 * m * (3 * h + it + 2 * h + 2 * kv + it + h)
        return {"bytes": params + 4 * rows + acts, "flops": 2 * m * params}
    if kind == "head":
        m, rows, k = case["m"], case["rows"], case["k"]
        es = 4 if case["dtype"] == "f32" else 2
        return {"bytes": rows * k + 4 * rows + m * (es * k + 12), "flops": 2 * m * rows * k}
    if kind == "w8a8":
        m, n, k = case["m"], case["n"], case["k"]
        es = 4 if case["out"] == "f32" else 2
        return {"bytes": n * k + 4 * n + 2 * m * k + es * m * n, "flops": 2 * m * n * k}
    if kind == "moe":
        T, E, top_k, H, inter = case["t"], case["experts"], case["top_k"], case["hidden"], case["inter"]
        # experts that T random top-k choices reach, on average
        active = E * (1.0 - (1.0 - top_k / E) ** T)
        page = 3 * H * inter + 4 * (2 * inter + H)
        return {"bytes": int(active * page) + T * (2 * E + 2 * 2 * H + 10 * top_k), "flops": 2 * T * top_k * 3 * H * inter}
    if kind == "lowbit":
        m, n, k, ng = case["m"], case["n"], case["k"], case["k"] // case["group"]
        es = 4 if case["dtype"] == "f32" else 2
        return {"bytes": n * k * case["bits"] // 8 + 4 * n * ng + es * m * k + 4 * m * n, "flops": 2 * m * n * k}
    n, k = case["n"], case["k"]
    ng = 1 if case["bits"] == 8 else -(-k // case["group"])
    # per weight: its magnitude, the running maximum or sum, the division and the rounding
    return {"bytes": 4 * n * k + n * k * case["bits"] // 8 + 4 * n * ng, "flops": 4 * n * k}


def tolerance(case: dict):
    kind = case["kind"]
    if kind == "encode":
        return "exact"
    if kind == "linear":
        # 32-bit sums of up to 8960 products; one rounding of the result to 16 bits
        return {"rel": {"f32": 2e-6, "bf16": 2e-3, "f16": 3e-4}[case["dtype"]]}
    if kind == "layer":
        return {"rel": 4e-3}  # bf16 results; act and down carry the gate and up roundings too
    if kind == "head":
        return {"rel": 2e-6, "differ": 0.0}
    if kind == "w8a8":
        return {"rel": 2e-6 if case["out"] == "f32" else 2e-3}
    if kind == "moe":
        return {"rel": 8e-3, "differ": 0.0}  # bf16 result over bf16 activations (requantized to int8 in W8A8)
    return {"rel": 2e-6}  # low-bit: fp32 sums and result


# ---- 64-bit results ------------------------------------------------------------------------


def _w16(w, dtype: torch.dtype) -> torch.Tensor:
    """The weight a product uses: one fp32 multiply, rounded to the activation dtype."""
    return (w[0].float() * w[1][:, None]).to(dtype).double()


def _silu_pair(g: torch.Tensor, u: torch.Tensor) -> torch.Tensor:
    """bf16(bf16(silu(bf16(g))) * bf16(u)) with each step in 64 bits."""
    g, u = g.bfloat16().double(), u.bfloat16().double()
    return ((g * torch.sigmoid(g)).bfloat16().double() * u).bfloat16().double()


def _act_quant(x: torch.Tensor, keep: torch.Tensor | None = None) -> tuple[torch.Tensor, torch.Tensor]:
    v = x.float() if keep is None else x.float() * keep
    s = v.abs().amax(dim=1) / 127.0
    s = torch.where(s == 0, torch.ones_like(s), s)
    return (v / s[:, None]).round().clamp(-127, 127).double(), s.double()


def exact(case: dict, seed: int):
    d = _inputs(case, seed)
    kind = case["kind"]
    if kind == "linear":
        return d["x"].double() @ _w16(d["w"], d["x"].dtype).t()
    if kind == "layer":
        bf = torch.bfloat16
        q, k, v = (d["x"].double() @ _w16(d[n], bf).t() for n in ("q", "k", "v"))
        o = d["attn"].double() @ _w16(d["o"], bf).t()
        mlp = d["mlp"].double()
        act = _silu_pair(mlp @ _w16(d["gate"], bf).t(), mlp @ _w16(d["up"], bf).t())
        return q, k, v, o, act, act @ _w16(d["down"], bf).t()
    if kind == "head":
        w = (d["w"][0][:case["rows"]], d["w"][1][:case["rows"]])
        x = d["x"].double()
        cand = torch.topk(x @ _w16(w, d["x"].dtype).t(), 2, dim=1).indices.sort(dim=1).values
        val = torch.stack([(_w16((w[0][c], w[1][c]), torch.float32) @ x[i]) for i, c in enumerate(cand)])
        best = val.argmax(dim=1, keepdim=True)
        return cand.gather(1, best)[:, 0], val.gather(1, best)[:, 0]
    if kind == "w8a8":
        x, (qw, sw) = d["x"], d["w"]
        side, keep = 0.0, None
        if case["protect"]:
            idx = torch.sort(x.float().abs().amax(dim=0), descending=True, stable=True).indices[:case["protect"]]
            keep = torch.ones(case["k"], device=DEV)
            keep[idx] = 0.0
            side = x[:, idx].double() @ (qw[:, idx].float() * sw[:, None]).double().t()
        q, s = _act_quant(x, keep)
        return side + (q @ qw.double().t()) * s[:, None] * sw.double()
    if kind == "moe":
        x = d["x"]
        p, order = torch.sort(torch.softmax(d["logits"].double(), dim=1), dim=1, descending=True, stable=True)
        w, experts = p[:, :case["top_k"]], order[:, :case["top_k"]]
        w = w / w.sum(dim=1, keepdim=True)
        w16 = w.bfloat16().double()
        xq, xs = _act_quant(x)
        out = torch.zeros(x.shape, dtype=torch.float64, device=DEV)
        inter = case["inter"]
        for e in range(case["experts"]):
            t, r = torch.nonzero(experts == e, as_tuple=True)
            if not t.numel():
                continue
            gu, gus, dn, dns = d["gate_up"][e], d["gate_up_scales"][e], d["down"][e], d["down_scales"][e]
            if case["w8a16"]:
                h = x[t].double() @ _w16((gu, gus), torch.bfloat16).t()
                act = _silu_pair(h[:, :inter], h[:, inter:])
                y = act @ _w16((dn, dns), torch.bfloat16).t()
            else:
                h = (xq[t] @ gu.double().t()) * xs[t, None] * gus.double()
                aq, as_ = _act_quant(_silu_pair(h[:, :inter], h[:, inter:]))
                y = (aq @ dn.double().t()) * as_[:, None] * dns.double()
            out.index_add_(0, t, y.bfloat16().double() * w16[t, r, None])
        return out, w, experts
    if kind == "lowbit":
        z = d["zeros"].float() if d["zeros"] is not None else (4.0 if case["bits"] == 3 else 1.0)
        c = d["codes"].float().view(case["n"], -1, case["group"])
        zz = z[:, :, None] if isinstance(z, torch.Tensor) else z
        w = ((c - zz) * d["scales"].float()[:, :, None]).double().view(case["n"], case["k"])
        return d["x"].double() @ w.t()
    if case["bits"] == 8:
        return None, d["w"].double().abs().amax(dim=1) / 127.0
    a = d["w"].double().abs().view(case["n"], -1, case["group"])
    if case["bits"] == 3:
        return None, a.amax(dim=2) / 3.0
    active = a >= 0.7 * a.mean(dim=2, keepdim=True)
    return None, (a * active).sum(dim=2) / active.sum(dim=2)
