"""The work whose time is tracked: GGUF quantized matmuls as an inference engine calls them.

The listed cases follow the engine's own calls on this path: decode GEMVs (one projection, a layer's four dependent
launches, all projections of a small model in one launch, the LM head), a few rows at once (small batches,
speculative tokens), prefill (attention projections, the fused FFN, a whole model's GEMMs, the 8-bit type at ragged
sizes), a mixture-of-experts layer in both directions, and the dequantization of a table. Sizes are those of
``reflex_amd.synth`` (Qwen3-0.6B, Qwen3-8B and Qwen3-MoE layers) or generic; ``draw`` spreads them.

Weights are raw GGUF blocks made on the GPU with codes and scales as a quantized network has them: codes about normal
around the block's centre, scales that put the weights at a standard deviation near 0.02. Activations are normal with
a few large channels, as a residual stream has them.
"""
import math

import torch

import reflex_amd as rq
from reflex_amd import synth

DEV = "cuda:0"
Q4K, Q6K, Q8_0 = synth.Q4K, synth.Q6K, synth.Q8_0
BLOCK = synth.BLOCK
TYPES = {"q4_k": Q4K, "q6_k": Q6K, "q8_0": Q8_0}

# sizes and weight types of one decoder layer (see _layer)
L06B = {"hidden": 1024, "q": 2048, "kv": 1024, "ffn": 3072, "mix": "q4_k_s"}
L8B = {"hidden": 4096, "q": 4096, "kv": 1024, "ffn": 14336, "mix": "q4_k_m"}
# the projections that one launch can hold: each group's inputs come from the group before
GROUPS = (("q_proj", "k_proj", "v_proj"), ("o_proj",), ("gate_proj", "up_proj"), ("down_proj",))
EPS = 1e-6


def listed():
    return [
        # the smallest call: one decode GEMV of an 8-bit file's square projection
        {"name": "gemv q8_0 1k", "kind": "gemv", "type": "q8_0", "n": 1024, "k": 1024},
        # one decode step's LM head, the largest single GEMV
        {"name": "gemv lm_head", "kind": "gemv", "type": "q6_k", "n": 151936, "k": 1024},
        # one decoder layer of a decode step: four dependent launches from kept plans
        {"name": "decode layer 8b", "kind": "decode_layer", **L8B},
        # every projection of the 0.6B model in one launch (the weights of a whole decode step)
        {"name": "decode set 0.6b", "kind": "decode_set", "layers": 28, **L06B},
        # a small batch or a run of speculative tokens through one layer
        {"name": "layer 8b 12 rows", "kind": "rows_layer", "rows": 12, **L8B},
        # prefill of an ordinary prompt: the attention projections of one layer, from f32 activations
        {"name": "attn 8b 512", "kind": "attn", "rows": 512, **L8B},
        # prefill of a long prompt: one layer's FFN through the fused producers (the largest case)
        {"name": "ffn 8b 2048", "kind": "ffn", "hidden": 4096, "ffn": 14336, "gate": "q4_k", "down": "q6_k",
         "rows": 2048},
        # prefill of an ordinary prompt through all projections of the 0.6B model, grouped
        {"name": "prefill set 0.6b 512", "kind": "prefill_set", "layers": 28, "rows": 512, **L06B},
        # an 8-bit file's projection at ragged sizes
        {"name": "gemm q8_0 ragged", "kind": "gemm", "type": "q8_0", "n": 4098, "k": 4096, "rows": 333},
        # a mixture-of-experts layer, prefill and decode, routed on the device
        {"name": "moe prefill 512", "kind": "moe", "experts": 128, "hidden": 2048, "ffn": 768, "top_k": 8,
         "rows": 512, "gate": "q4_k", "down": "q4_k", "route": "device"},
        {"name": "moe decode", "kind": "moe", "experts": 128, "hidden": 2048, "ffn": 768, "top_k": 8,
         "rows": 1, "gate": "q4_k", "down": "q4_k", "route": "device"},
        # a quantized embedding table turned into f16
        {"name": "dequantize table", "kind": "dequantize", "type": "q6_k", "n": 151936, "k": 1024, "out": "f16"},
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _unit(rng, lo, hi):
    """A multiple of 256 between lo and hi, over the logarithm."""
    return 256 * max(1, _log(rng, lo / 256, hi / 256))


def _draw_layer(rng):
    hidden = _unit(rng, 1024, 4096)
    return {"hidden": hidden, "q": _unit(rng, hidden, min(2 * hidden, 4096)), "kv": 128 * rng.randint(2, 8),
            "ffn": _unit(rng, 2 * hidden, 3.5 * hidden), "mix": rng.choice(["q4_k_s", "q4_k_m", "q4_k_m", "q8_0"])}


def draw(rng):
    kind = rng.choice(["gemv", "gemv", "decode_layer", "rows_layer", "gemm", "gemm", "gemm", "attn", "ffn", "ffn",
                       "moe", "moe", "dequantize"])
    ty = rng.choice(["q4_k", "q4_k", "q6_k", "q8_0"])
    if kind == "gemv":
        k = _unit(rng, 256, 14336)
        return {"kind": kind, "type": ty, "n": _log(rng, 64, min(151936, 150_000_000 // k)), "k": k}
    if kind == "decode_layer":
        return {"kind": kind, **_draw_layer(rng)}
    if kind == "rows_layer":
        return {"kind": kind, "rows": _log(rng, 2, 96), **_draw_layer(rng)}
    if kind == "gemm":
        rows = _log(rng, 2, 2048)
        k = _unit(rng, 256, 14336)
        return {"kind": kind, "type": ty, "n": _log(rng, 256, min(32768, 150_000_000_000 // (rows * k))), "k": k,
                "rows": rows}
    if kind == "attn":
        return {"kind": kind, "rows": _log(rng, 24, 2048), **_draw_layer(rng)}
    if kind == "ffn":
        hidden = _unit(rng, 1024, 4096)
        return {"kind": kind, "hidden": hidden, "ffn": _unit(rng, hidden, 3.5 * hidden),
                "gate": rng.choice(["q4_k", "q4_k", "q8_0"]), "down": rng.choice(["q4_k", "q6_k", "q8_0"]),
                "rows": _log(rng, 16, 2048)}
    if kind == "moe":
        experts = rng.choice([8, 32, 64, 128])
        return {"kind": kind, "experts": experts, "hidden": _unit(rng, 1024, 4096), "ffn": _unit(rng, 512, 1536),
                "top_k": rng.randint(2, 8), "rows": _log(rng, 1, 1024), "gate": "q4_k",
                "down": rng.choice(["q4_k", "q6_k"]), "route": rng.choice(["device", "device", "device", "host"])}
    k = _unit(rng, 256, 14336)
    return {"kind": kind, "type": ty, "n": _log(rng, 256, 150_000_000 // k), "k": k, "out": rng.choice(["f16", "f32"])}


# ---------------------------------------------------------------- inputs

class _Maker:
    """Tensors from one seed, in the order asked for."""

    def __init__(self, seed):
        self.gen = torch.Generator(device=DEV)
        self.gen.manual_seed(seed)

    def normal(self, *shape):
        return torch.randn(*shape, device=DEV, generator=self.gen)

    def uniform(self, *shape):
        return torch.rand(*shape, device=DEV, generator=self.gen)

    def acts(self, rows, k):
        """Normal activations, one channel in 256 eight times as large."""
        big = torch.ones(k, device=DEV)
        big[torch.randperm(k, device=DEV, generator=self.gen)[: max(1, k // 256)]] = 8.0
        return (self.normal(rows, k) * big).reshape(-1)

    def blocks(self, ty, rows, k):
        """Raw blocks of a [rows][k] weight, made in pieces of about 16 M values."""
        qk, bb = BLOCK[ty]
        per = k // qk
        out = torch.empty(rows * per, bb, dtype=torch.uint8, device=DEV)
        step = max(1, (1 << 24) // k) * per
        for i in range(0, rows * per, step):
            out[i:i + step] = self._piece(ty, min(step, rows * per - i))
        return out.reshape(-1)

    def _codes(self, n, m, spread, centre, top):
        return (self.normal(n, m) * spread + centre).round_().clamp_(0, top).to(torch.uint8)

    def _half(self, n, size):
        """f16 scales about `size`, as bytes."""
        return (size * (0.7 + 0.6 * self.uniform(n, 1))).half().view(torch.uint8)

    def _piece(self, ty, n):
        if ty == Q8_0:
            q = (self.normal(n, 32) * 42.0).round_().clamp_(-127, 127).to(torch.int8).view(torch.uint8)
            return torch.cat([self._half(n, 0.02 / 42.0), q], 1)
        if ty == Q4K:
            # w = d sc q - dmin m with dmin = 8 d and m near sc: about d sc (q - 8)
            d = (0.02 / (2.8 * 45.0)) * (0.7 + 0.6 * self.uniform(n, 1))
            sc = (28.0 + 35.0 * self.uniform(n, 8)).to(torch.uint8)
            m = (sc.float() * (0.9 + 0.2 * self.uniform(n, 8))).round_().clamp_(0, 63).to(torch.uint8)
            head = torch.cat([(sc[:, :4] & 63) | ((sc[:, 4:] >> 4) << 6), (m[:, :4] & 63) | ((m[:, 4:] >> 4) << 6),
                              (sc[:, 4:] & 15) | ((m[:, 4:] & 15) << 4)], 1)
            q = self._codes(n, 256, 2.8, 8.0, 15).view(n, 4, 2, 32)
            return torch.cat([d.half().view(torch.uint8), (8.0 * d).half().view(torch.uint8), head,
                              (q[:, :, 0] | (q[:, :, 1] << 4)).reshape(n, 128)], 1)
        q = self._codes(n, 256, 10.0, 32.0, 63).view(n, 2, 4, 32)  # half, group, position
        low, high = q & 15, q >> 4
        ql = torch.cat([low[:, :, 0] | (low[:, :, 2] << 4), low[:, :, 1] | (low[:, :, 3] << 4)], 2)
        qh = high[:, :, 0] | (high[:, :, 1] << 2) | (high[:, :, 2] << 4) | (high[:, :, 3] << 6)
        sign = 1.0 - 2.0 * (self.uniform(n, 16) < 0.5).float()
        sc = ((40.0 + 87.0 * self.uniform(n, 16)) * sign).round_().to(torch.int8).view(torch.uint8)
        return torch.cat([ql.reshape(n, 128), qh.reshape(n, 64), sc, self._half(n, 0.02 / (10.0 * 80.0))], 1)

    def weight(self, ty, n, k, experts=0):
        b = self.blocks(ty, n * max(1, experts), k)
        return rq.Weight(rq.GgmlType(ty), b, [k, n] + ([experts] if experts else []))


def _layer(case):
    """{projection: (type, out, in)} of the case's layer: Q4_K with Q6_K for v and perhaps down, or all Q8_0."""
    h, q, kv, ffn = (case[m] for m in ("hidden", "q", "kv", "ffn"))
    most, v, down = {"q4_k_s": (Q4K, Q6K, Q4K), "q4_k_m": (Q4K, Q6K, Q6K), "q8_0": (Q8_0, Q8_0, Q8_0)}[case["mix"]]
    return {"q_proj": (most, q, h), "k_proj": (most, kv, h), "v_proj": (v, kv, h), "o_proj": (most, h, q),
            "gate_proj": (most, ffn, h), "up_proj": (most, ffn, h), "down_proj": (down, h, ffn)}


def _layer_state(case, mk, rows):
    """One layer's weights, the input of each group of projections and every output."""
    layer = _layer(case)
    w = {p: mk.weight(ty, n, k) for p, (ty, n, k) in layer.items()}
    x = {g: mk.acts(rows, layer[g[0]][2]) for g in GROUPS}
    y = {p: torch.empty(rows * n, device=DEV) for p, (_, n, _) in layer.items()}
    return w, x, y


def _set_state(case, mk, rows):
    """Every layer's (input, weight, output) triples and all outputs in one tensor."""
    layer, items, at = _layer(case), [], 0
    y = torch.empty(rows * case["layers"] * sum(n for _, n, _ in layer.values()), device=DEV)
    for _ in range(case["layers"]):
        for g in GROUPS:
            x = mk.acts(rows, layer[g[0]][2])
            for p in g:
                ty, n, k = layer[p]
                items.append((x, mk.weight(ty, n, k), y[at:at + rows * n]))
                at += rows * n
    return items, y


def prepare(case, seed):
    mk, kind = _Maker(seed), case["kind"]
    s = {"case": case}
    if kind == "gemv":
        s["w"] = mk.weight(TYPES[case["type"]], case["n"], case["k"])
        s["x"] = mk.acts(1, case["k"])
        s["y"] = torch.empty(case["n"], device=DEV)
    elif kind == "decode_layer":
        s["w"], s["x"], s["y"] = _layer_state(case, mk, 1)
        s["plans"] = [rq.GemvPlan([(s["x"][g], s["w"][p], s["y"][p]) for p in g]) for g in GROUPS]
    elif kind == "decode_set":
        items, s["y"] = _set_state(case, mk, 1)
        s["plan"] = rq.GemvPlan(items)
    elif kind == "rows_layer":
        s["w"], s["x"], s["y"] = _layer_state(case, mk, case["rows"])
        s["plans"] = [rq.GemmPlan([(s["x"][g], s["w"][p], s["y"][p]) for p in g], case["rows"]) for g in GROUPS]
    elif kind == "attn":
        s["w"], s["x"], s["y"] = _layer_state(case, mk, case["rows"])
    elif kind == "prefill_set":
        items, s["y"] = _set_state(case, mk, case["rows"])
        s["plan"] = rq.GemmPlan(items, case["rows"])
    elif kind == "gemm":
        s["w"] = mk.weight(TYPES[case["type"]], case["n"], case["k"])
        s["x"] = mk.acts(case["rows"], case["k"])
        s["y"] = torch.empty(case["rows"] * case["n"], device=DEV)
    elif kind == "ffn":
        h, f = case["hidden"], case["ffn"]
        s["gate"], s["up"] = (mk.weight(TYPES[case["gate"]], f, h) for _ in range(2))
        s["down"] = mk.weight(TYPES[case["down"]], h, f)
        s["norm"] = 1.0 + 0.1 * mk.normal(h)
        s["x"] = mk.acts(case["rows"], h)
        s["y"] = torch.empty(case["rows"] * h, device=DEV)
    elif kind == "moe":
        h, f, e = case["hidden"], case["ffn"], case["experts"]
        s["gate"], s["up"] = (mk.weight(TYPES[case["gate"]], f, h, e) for _ in range(2))
        s["down"] = mk.weight(TYPES[case["down"]], h, f, e)
        s["x"] = mk.acts(case["rows"], h)
        s["logits"] = mk.normal(case["rows"], e)
        if case["route"] == "host":  # the engine has copied them there
            s["logits"] = s["logits"].cpu().numpy()
        s["y"] = torch.empty(case["rows"] * h, device=DEV)
    elif kind == "dequantize":
        s["blocks"] = mk.blocks(TYPES[case["type"]], case["n"], case["k"])
    else:
        raise ValueError(kind)
    return s


# ---------------------------------------------------------------- one pass

def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "gemv":
        rq.gemv_to(s["x"], s["w"], s["y"])
    elif kind in ("decode_layer", "rows_layer"):
        for p in s["plans"]:
            p.run()
    elif kind in ("decode_set", "prefill_set"):
        s["plan"].run()
    elif kind == "attn":
        g = GROUPS[0]
        rq.gemm_batch([(s["x"][g], s["w"][p], s["y"][p]) for p in g], case["rows"])
        rq.gemm(s["x"][GROUPS[1]], s["w"]["o_proj"], case["rows"], out=s["y"]["o_proj"])
        return {p: s["y"][p] for p in (*g, "o_proj")}
    elif kind == "gemm":
        rq.gemm(s["x"], s["w"], case["rows"], out=s["y"])
    elif kind == "ffn":
        act, _ = rq.rmsnorm_q8_1(s["x"], s["norm"], case["rows"], case["hidden"], EPS)
        act, inner = rq.gemm_gate_up_silu_q8_1(act, case["rows"], s["gate"], s["up"])
        rq.gemm_q8_1(act, s["down"], case["rows"], out=s["y"])
        return {"inner": inner, "y": s["y"]}
    elif kind == "moe":
        ffn = rq.moe_ffn_grouped if case["route"] == "host" else rq.moe_ffn_grouped_device
        ffn(s["x"], case["rows"], case["hidden"], s["logits"], case["experts"], case["top_k"], True, 1.0, s["gate"],
            s["up"], s["down"], s["y"])
    else:
        return rq.dequantize(TYPES[case["type"]], s["blocks"], case["n"] * case["k"],
                             torch.float16 if case["out"] == "f16" else torch.float32)
    return s["y"]


# ---------------------------------------------------------------- what a pass cannot do without

def _matmul(ty, n, k, rows):
    """(bytes of the weights and the outputs, operations)."""
    return synth.weight_bytes(ty, n, k) + 4 * rows * n, 2 * rows * n * k


def work(case):
    kind = case["kind"]
    if kind == "dequantize":
        count = case["n"] * case["k"]
        return {"bytes": synth.weight_bytes(TYPES[case["type"]], case["n"], case["k"])
                + count * (2 if case["out"] == "f16" else 4), "flops": 2 * count}
    if kind == "ffn":
        h, f, rows = case["hidden"], case["ffn"], case["rows"]
        parts = [_matmul(TYPES[case["gate"]], f, h, rows)] * 2 + [_matmul(TYPES[case["down"]], h, f, rows)]
        # gate and up give one output between them
        return {"bytes": sum(p[0] for p in parts) - 4 * rows * f + 4 * rows * h + 4 * h,
                "flops": sum(p[1] for p in parts)}
    if kind == "moe":
        h, f, rows, e, k = case["hidden"], case["ffn"], case["rows"], case["experts"], case["top_k"]
        used = e * (1.0 - (1.0 - k / e) ** rows)  # experts that get a row, on average
        one = 2 * synth.weight_bytes(TYPES[case["gate"]], f, h) + synth.weight_bytes(TYPES[case["down"]], h, f)
        return {"bytes": used * one + 4 * rows * (2 * h + e), "flops": 2 * rows * k * 3 * h * f}
    if kind in ("gemv", "gemm"):
        rows = case.get("rows", 1)
        b, ops = _matmul(TYPES[case["type"]], case["n"], case["k"], rows)
        return {"bytes": b + 4 * rows * case["k"], "flops": ops}
    layer = _layer(case)
    rows, count = case.get("rows", 1), case.get("layers", 1)
    groups = GROUPS[:2] if kind == "attn" else GROUPS
    parts = [_matmul(*layer[p], rows) for g in groups for p in g]
    return {"bytes": count * (sum(p[0] for p in parts) + sum(4 * rows * layer[g[0]][2] for g in groups)),
            "flops": count * sum(p[1] for p in parts)}


def tolerance(case):
    """Dequantization is defined to the bit. The products take f16 operands: against 64 bits the activations' rounding
    alone shows about 2.1e-4 (GEMVs), with the weight operands' 3.5e-4 (tiles), two products in a row 6.1e-4; another
    f16 implementation is as far off again, in another direction. About four times these."""
    kind = case["kind"]
    if kind == "dequantize":
        return "exact"
    if kind in ("ffn", "moe"):
        return {"rel": 2.4e-3, "max": 2.4e-2}
    if kind in ("gemv", "decode_layer", "decode_set"):
        return {"rel": 8e-4, "max": 8e-3}
    return {"rel": 1.4e-3, "max": 1.4e-2}


# ---------------------------------------------------------------- the same in 64 bits

def _values(ty, blocks, n, k):
    """The weights [n][k] that raw blocks stand for, in f64."""
    qk, bb = BLOCK[ty]
    b = blocks.view(-1, bb)

    def half(lo):
        return b[:, lo:lo + 2].contiguous().view(torch.float16).double()

    if ty == Q8_0:
        w = half(0) * b[:, 2:34].contiguous().view(torch.int8).double()
    elif ty == Q4K:
        s, m, t = b[:, 4:8], b[:, 8:12], b[:, 12:16]
        sc = torch.cat([s & 63, (t & 15) | ((s >> 6) << 4)], 1).double()
        mn = torch.cat([m & 63, (t >> 4) | ((m >> 6) << 4)], 1).double()
        qs = b[:, 16:144].view(-1, 4, 1, 32)
        q = torch.cat([qs & 15, qs >> 4], 2).view(-1, 8, 32).double()
        w = (half(0) * sc)[:, :, None] * q - (half(2) * mn)[:, :, None]
    else:
        ql, qh = b[:, :128].view(-1, 2, 2, 32), b[:, 128:192].view(-1, 2, 1, 32)
        low = torch.cat([ql & 15, ql >> 4], 2)
        high = torch.cat([(qh >> s) & 3 for s in (0, 2, 4, 6)], 2)
        q = (low | (high << 4)).double() - 32.0
        sc = b[:, 192:208].contiguous().view(torch.int8).double()
        w = (half(208) * sc)[:, :, None] * q.view(-1, 16, 16)
    return w.reshape(n, k)


def _product(x, w, rows):
    """x [rows][k] . W^T in f64, a piece of the weight's rows at a time."""
    k, n = w.in_features, w.out_features
    rb = w.len // n
    x = x.view(rows, k).double()
    y = torch.empty(rows, n, dtype=torch.float64, device=DEV)
    blocks = w.arena[w.offset:w.offset + w.len]
    step = max(1, (1 << 26) // k)
    for i in range(0, n, step):
        m = min(step, n - i)
        y[:, i:i + m] = x @ _values(int(w.ty), blocks[i * rb:(i + m) * rb], m, k).t().contiguous()
    return y


def _silu_mul(g, u):
    return g * torch.sigmoid(g) * u


def exact(case, seed):
    s, kind = prepare(case, seed), case["kind"]
    if kind in ("gemv", "gemm"):
        return _product(s["x"], s["w"], case.get("rows", 1)).reshape(-1)
    if kind in ("decode_layer", "rows_layer", "attn"):
        groups = GROUPS[:2] if kind == "attn" else GROUPS
        return {p: _product(s["x"][g], s["w"][p], case.get("rows", 1)).reshape(-1) for g in groups for p in g}
    if kind in ("decode_set", "prefill_set"):
        items, _ = _set_state(case, _Maker(seed), case.get("rows", 1))
        return torch.cat([_product(x, w, case.get("rows", 1)).reshape(-1) for x, w, _ in items])
    if kind == "ffn":
        x = s["x"].view(case["rows"], -1).double()
        x = x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS) * s["norm"].double()
        inner = _silu_mul(_product(x, s["gate"], case["rows"]), _product(x, s["up"], case["rows"]))
        return {"inner": inner.reshape(-1), "y": _product(inner, s["down"], case["rows"]).reshape(-1)}
    if kind == "moe":
        x = s["x"].view(case["rows"], -1).double()
        p = torch.softmax(torch.as_tensor(s["logits"]).to(DEV).double(), 1)
        top, idx = torch.topk(p, case["top_k"], dim=1)
        top = top / top.sum(1, keepdim=True)
        y = torch.zeros_like(x)
        for e in range(case["experts"]):
            row, slot = torch.nonzero(idx == e, as_tuple=True)
            if row.numel():
                gate, up, down = (rq.quant_expert_weight(s[m], e) for m in ("gate", "up", "down"))
                n = row.numel()
                inner = _silu_mul(_product(x[row], gate, n), _product(x[row], up, n))
                y.index_add_(0, row, _product(inner, down, n) * top[row, slot][:, None])
        return y.reshape(-1)
    return _values(TYPES[case["type"]], s["blocks"], case["n"], case["k"]).reshape(-1)
