"""Performance cases of the MoE forward and the segmented-KV GQA attention.

Each case is one call of a public entry point as a serving program makes it:
the operator is prepared once on buffers that stay in place (weights, plan,
owned output), and a pass is one forward on the current stream.

The MoE shapes are the Qwen3-30B-A3B layer (E 128, H 2048, I 768, top-8), one
GPU's share of it under 8-way expert parallelism (16 experts, one route per
received row) and under 8-way tensor parallelism (I 96), and a layer whose
dimensions are not powers of two (E 32, H = I = 2880, top-4).  Decode batches
are 1 to a few hundred tokens, prefill chunks up to 4096.  The attention is
the prefill of a chunk of T tokens against three cached history segments.
"""
import math

import torch

from llm_gpu_kernels_amd import TiledGateUp, prepare_moe, prepare_routed_moe, prepare_segmented_gqa, prepare_w4_moe

QWEN = dict(E=128, H=2048, I=768, K=8)
EP8 = dict(E=16, H=2048, I=768, K=1)
TP8 = dict(E=128, H=2048, I=96, K=8)
WIDE = dict(E=32, H=2880, I=2880, K=4)
GROUP = 128  # W4 quantisation group along the hidden dimension


def _moe(name, dims, tokens, weights="bf16", routing="uniform", entry="routed"):
    case = dict(kind="moe", T=tokens, weights=weights, routing=routing, entry=entry, **dims)
    return dict(case, name=name) if name else case


def _gqa(name, tokens, history, heads=32, kv_heads=8, v_stride=0):
    case = dict(kind="gqa", T=tokens, h0=history[0], h1=history[1], h2=history[2], Hq=heads, Hkv=kv_heads,
                v_stride=v_stride)
    return dict(case, name=name) if name else case


def listed():
    return [
        # One sequence decoding: the smallest call, launches and latency count.
        _moe("bf16-t1", QWEN, 1),
        # A small decode batch, about one row per expert.
        _moe("bf16-t17", QWEN, 17),
        # A large decode batch: a dozen ragged rows per expert.
        _moe("bf16-t193", QWEN, 193),
        # A prefill chunk with skewed routing: a few experts take most rows.
        _moe("bf16-t1024-zipf", QWEN, 1024, routing="zipf"),
        # The largest prefill chunk.
        _moe("bf16-t4096", QWEN, 4096),
        # The small decode batch on int4 gate/up weights.
        _moe("w4-t17", QWEN, 17, weights="w4"),
        # A prefill chunk on int4 gate/up weights.
        _moe("w4-t1024", QWEN, 1024, weights="w4"),
        # A large ragged prefill chunk on int4 gate/up weights, skewed routing.
        _moe("w4-t3001-zipf", QWEN, 3001, weights="w4", routing="zipf"),
        # A layer of other dimensions, routes given by the caller as int64 ids.
        _moe("bf16-wide-t512-fixed", WIDE, 512, entry="fixed"),
        # Attention of a short, an ordinary and a long prefill chunk; the last
        # on ragged segments whose values lie in a wider cache row.
        _gqa("gqa-t32", 32, (1024, 512, 256)),
        _gqa("gqa-t256", 256, (1024, 512, 256)),
        _gqa("gqa-t2048-long", 2048, (8192, 2049, 575), v_stride=6144),
    ]


def _log_int(rng, low, high):
    return min(high, max(low, round(math.exp(rng.uniform(math.log(low), math.log(high))))))


def draw(rng):
    if rng.random() < 0.3:
        heads, kv = rng.choice([(32, 8), (32, 8), (16, 8), (8, 8)])
        history = (_log_int(rng, 16, 8192), rng.choice([0, _log_int(rng, 1, 2049)]), _log_int(rng, 1, 575))
        return _gqa(None, _log_int(rng, 1, 2048), history, heads, kv, rng.choice([0, 6144]))
    dims, most = rng.choice([(QWEN, 4096)] * 4 + [(EP8, 4096), (TP8, 4096), (WIDE, 1024)])
    weights = "bf16" if dims is WIDE else rng.choice(["bf16", "bf16", "w4", "w4fold"])
    routing = rng.choice(["uniform", "zipf"])
    entry = "fixed" if weights != "w4fold" and rng.random() < 0.25 else "routed"
    return _moe(None, dims, _log_int(rng, 1, most), weights, routing, entry)


# ---- inputs -----------------------------------------------------------------


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _randn_bf16(shape, gen, scale=1.0):
    """N(0, scale) in bf16, made in pieces along the first dimension."""
    out = torch.empty(shape, dtype=torch.bfloat16, device="cuda")
    rows = max(1, (1 << 27) // max(1, math.prod(shape[1:])))
    for i in range(0, shape[0], rows):
        part = out[i:i + rows]
        part.copy_(torch.randn(part.shape, generator=gen, device="cuda") * scale)
    return out


def _quantised(case, gen):
    """Symmetric int4 gate/up weights: q in [-7, 7] as int8 [E, 2I, H] and bf16
    scales [E, 2I, H / 128], from N(0, 0.02) weights."""
    e, n, k = case["E"], 2 * case["I"], case["H"]
    q = torch.empty((e, n, k), dtype=torch.int8, device="cuda")
    scales = torch.empty((e, n, k // GROUP), dtype=torch.bfloat16, device="cuda")
    for i in range(e):
        w = torch.randn((n, k // GROUP, GROUP), generator=gen, device="cuda") * 0.02
        s = (w.abs().amax(-1) / 7).to(torch.bfloat16)
        scales[i] = s
        q[i] = (w / s.float()[..., None]).round().clamp(-7, 7).to(torch.int8).view(n, k)
    return q, scales


def _tiled(q, scales):
    """The prepared W4 layout that a program loads: words [E, N/16, K/128, 64
    lanes, 4] (lane 16 g + r: row r, chunks of 8 K values at 8 g + 32 j, low
    nibble first) and scales [E, N/16, K/128, 16]."""
    e, n, k = q.shape
    words = torch.empty((e, n // 16, k // GROUP, 64, 4), dtype=torch.int32, device=q.device)
    for i in range(e):
        nib = (q[i].view(n // 16, 16, k // GROUP, 4, 4, 8).to(torch.int64) + 8)
        packed = torch.zeros(nib.shape[:-1], dtype=torch.int64, device=q.device)
        for b in range(8):
            packed |= nib[..., b] << (4 * b)
        packed = torch.where(packed >= 2 ** 31, packed - 2 ** 32, packed).to(torch.int32)
        # [N/16, row, K/128, j, g] -> [N/16, K/128, g, row, j]
        words[i] = packed.permute(0, 2, 4, 1, 3).reshape(n // 16, k // GROUP, 64, 4)
    st = scales.view(e, n // 16, 16, k // GROUP).transpose(2, 3).contiguous()
    return TiledGateUp(words, st, (e, n, k))


def _moe_inputs(case, seed):
    gen = _generator(seed)
    t, e, h, inter = case["T"], case["E"], case["H"], case["I"]
    x = _randn_bf16((t, h), gen)
    logits = torch.randn((t, e), generator=gen, device="cuda")
    if case["routing"] == "zipf":
        rank = torch.arange(1, e + 1, dtype=torch.float32, device="cuda")
        bias = torch.empty(e, device="cuda")
        bias[torch.randperm(e, generator=gen, device="cuda")] = -1.2 * rank.log()
        logits = logits + bias
    down = _randn_bf16((e, h, inter), gen, 0.02)
    if case["weights"] == "bf16":
        gate_up = _randn_bf16((e, 2 * inter, h), gen, 0.02)
    else:
        gate_up = _quantised(case, gen)
    return x, logits.contiguous(), gate_up, down


def _top_k(logits, k):
    """The k largest logits per token (ties to the lower expert) and their
    softmax weights, renormalised, in the logits' type."""
    ids = logits.sort(dim=-1, descending=True, stable=True).indices[:, :k]
    return ids, torch.softmax(logits.gather(1, ids), dim=-1)


def _gqa_inputs(case, seed):
    gen = _generator(seed)
    t, hq, hkv = case["T"], case["Hq"], case["Hkv"]
    q = _randn_bf16((t, hq, 128), gen)
    segments = []
    for length in (case["h0"], case["h1"], case["h2"], t):
        k = _randn_bf16((length, hkv, 128), gen)
        if case["v_stride"]:
            v = _randn_bf16((length, case["v_stride"]), gen)[:, :hkv * 128].unflatten(1, (hkv, 128))
        else:
            v = _randn_bf16((length, hkv, 128), gen)
        segments.append((k, v))
    return q, segments


# ---- one pass -----------------------------------------------------------------


def prepare(case, seed):
    if case["kind"] == "gqa":
        q, segments = _gqa_inputs(case, seed)
        return dict(entry="gqa", plan=prepare_segmented_gqa(q, segments))
    x, logits, gate_up, down = _moe_inputs(case, seed)
    if case["weights"] != "bf16":
        gate_up = _tiled(*gate_up)
    if case["entry"] == "fixed":
        ids, weights = _top_k(logits, case["K"])
        if case["weights"] == "bf16":
            plan = prepare_moe(x, gate_up, down, ids.contiguous(), weights.contiguous())
        else:
            plan = prepare_w4_moe(x, gate_up, down, ids.contiguous(), weights.contiguous())
        return dict(entry="fixed", plan=plan)
    plan = prepare_routed_moe(x, logits, gate_up, down, case["K"],
                              w4_decode="fold" if case["weights"] == "w4fold" else "exact")
    return dict(entry="routed", plan=plan, x=x, logits=logits)


def run(state):
    plan = state["plan"]
    if state["entry"] != "routed":
        return plan.run()
    out = plan.forward(state["x"], state["logits"])
    return dict(out=out, ids=plan.ids, weights=plan.routing_weights)


# ---- what a pass cannot do without ----------------------------------------------


def work(case):
    t, bf16 = case["T"], 2
    if case["kind"] == "gqa":
        history = case["h0"] + case["h1"] + case["h2"]
        hq, hkv = case["Hq"], case["Hkv"]
        return dict(bytes=(history + t) * hkv * 128 * 2 * bf16 + 2 * t * hq * 128 * bf16,
                    flops=hq * 4 * 128 * (t * history + t * (t + 1) // 2))
    e, h, inter, k = case["E"], case["H"], case["I"], case["K"]
    r = t * k
    if case["routing"] == "zipf":
        # Experts with a row, of routes drawn like the inputs' (the
        # permutation of the experts does not matter here).
        logits = torch.randn((t, e), generator=torch.Generator().manual_seed(0))
        logits -= 1.2 * torch.arange(1, e + 1, dtype=torch.float32).log()
        active = len(logits.topk(k, dim=-1).indices.unique())
    else:
        active = e * (1 - (1 - k / e) ** t)
    gate_up = 2 * inter * h * bf16 if case["weights"] == "bf16" else 2 * inter * (h // 2 + h // GROUP * bf16)
    id_bytes = 8 if case["entry"] == "fixed" else 4
    route = r * (id_bytes + 4) + (t * e * 4 if case["entry"] == "routed" else 0)
    return dict(bytes=int(active * (gate_up + h * inter * bf16)) + 2 * t * h * bf16 + route,
                flops=6 * r * h * inter)


def tolerance(case):
    """MoE: gate, up, the SwiGLU product, each down row and the output are
    rounded to bf16 (2^-9 each).  Sums in another order move some of them to
    the neighbouring value: 2.7e-4 in norm and 1.5e-2 at most between two
    kernel families; against 64-bit sums without those roundings the path is
    3.9e-3 off, 2.9e-2 at most.  Attention: probabilities and the output are
    rounded to bf16, 2.3e-3 off and 1.2e-2 at most, and a probability's
    rounding depends on the reference maximum.  Router ids are the same."""
    return {"rel": 5e-3, "max": 6e-2, "differ": 0.0}


# ---- the same in 64 bits ----------------------------------------------------------


def _exact_gqa(case, seed):
    q, segments = _gqa_inputs(case, seed)
    t, hq, hkv = case["T"], case["Hq"], case["Hkv"]
    group = hq // hkv
    keys = torch.cat([k for k, _ in segments])
    values = torch.cat([v for _, v in segments])
    history = keys.shape[0] - t
    out = torch.empty((t, hq, 128), dtype=torch.float64, device="cuda")
    cols = torch.arange(keys.shape[0], device="cuda")
    rows = max(1, (1 << 27) // (group * keys.shape[0]))
    for j in range(hkv):
        kj, vj = keys[:, j].double(), values[:, j].double()
        for i in range(0, t, rows):
            qi = q[i:i + rows, j * group:(j + 1) * group].double()
            n = qi.shape[0]
            s = (qi.reshape(-1, 128) @ kj.t().contiguous()).view(n, group, -1) / math.sqrt(128.0)
            last = history + torch.arange(i, i + n, device="cuda")
            s.masked_fill_((cols > last[:, None])[:, None, :], -math.inf)
            p = torch.softmax(s, dim=-1)
            out[i:i + n, j * group:(j + 1) * group] = (p.view(n * group, -1) @ vj).view(n, group, 128)
    return out


def _exact_moe(case, seed):
    x, logits, gate_up, down = _moe_inputs(case, seed)
    inter, k = case["I"], case["K"]
    ids, weights = _top_k(logits.double(), k)
    if case["entry"] == "fixed":
        weights = _top_k(logits, k)[1].double()  # the weights that the call is given
    out = torch.zeros(x.shape, dtype=torch.float64, device="cuda")
    for e in range(case["E"]):
        token, slot = (ids == e).nonzero(as_tuple=True)
        if not len(token):
            continue
        if case["weights"] == "bf16":
            w = gate_up[e].double()
        else:
            q, scales = gate_up[0][e], gate_up[1][e]
            w = q.view(q.shape[0], -1, GROUP).double() * scales.double()[..., None]
            if case["weights"] == "w4":  # the weights are the products rounded to bf16
                w = w.to(torch.bfloat16).double()
            w = w.view(q.shape)
        y = x[token].double() @ w.t().contiguous()
        g, u = y[:, :inter], y[:, inter:]
        rows = (g / (1 + torch.exp(-g)) * u) @ down[e].double().t().contiguous()
        out.index_add_(0, token, rows * weights[token, slot][:, None])
    if case["entry"] == "fixed":
        return out
    return dict(out=out, ids=ids.to(torch.int32), weights=weights)


def exact(case, seed):
    return _exact_gqa(case, seed) if case["kind"] == "gqa" else _exact_moe(case, seed)
