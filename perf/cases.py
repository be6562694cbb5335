"""The work that this package is measured on: what a serving program has it do.

Each case is one call of a public entry point on data that is already on the
GPU, at the sizes of the package's own configurations: the MoE FFN block and
sub-layer from one decode token to a 4096-token prefill batch (fp32, bf16, fp8
weights, fp8 activations), ``mul_mat_id`` on its own, and the decode step's
attention half over a paged KV cache.

``listed()`` holds the named cases, ``draw(rng)`` one more of the same ranges.
``prepare`` makes the inputs and the object a program keeps (packed weights and
a workspace), ``run`` is one call, ``exact`` the same result in 64 bits from
plain torch.
"""

from __future__ import annotations

import importlib
import math

import torch

fm = importlib.import_module("frank-models_amd")

# name: n_embd, n_ff, n_expert, n_expert_used, normalize, router margin, Zipf exponent of the routing
MODELS = {
    "toy": (64, 128, 8, 2, True, 1e-6, 0.0),
    "mixtral": (4096, 14336, 8, 2, False, 1e-3, 0.0),
    "qwen3": (2048, 768, 128, 8, True, 1e-4, 1.1),
    "deepseek": (2048, 1408, 64, 6, False, 1e-4, 0.0),
}
# Largest batch of a drawn block: the configurations' largest prefill batch,
# and in fp32 one that costs no more than the largest listed case.
MAX_TOKENS = {"toy": 4096, "mixtral": 4096, "qwen3": 8192, "deepseek": 8192}
MAX_TOKENS_F32 = {"toy": 4096, "deepseek": 500}

# name: n_embd, n_head, n_head_kv
ATTENTION = {"mixtral": (4096, 32, 8), "small": (512, 4, 2)}

TORCH = {"bf16": torch.bfloat16, "f32": torch.float32}
BYTES = {"bf16": 2, "f32": 4, "fp8": 1}
EPS = 1e-5


def _block(name, model, tokens, form="block", act="bf16", weights="bf16", fp8_act="none"):
    return {"name": name, "kind": "block", "form": form, "model": model, "tokens": tokens, "act": act,
            "weights": weights, "fp8_act": fp8_act}


def _mmid(name, model, proj, tokens, act="bf16"):
    return {"name": name, "kind": "mul_mat_id", "model": model, "proj": proj, "tokens": tokens, "act": act}


def _attention(name, model, batch, context, ragged, bias, act="bf16", weights="bf16", block_size=16):
    return {"name": name, "kind": "attention", "model": model, "batch": batch, "context": context,
            "ragged": ragged, "bias": bias, "act": act, "weights": weights, "block_size": block_size}


def listed():
    return [
        # The drop-in function in the reference's own type at its toy model's
        # size: what a first user runs, all launches and host work.
        _block("toy-f32-32", "toy", 32, form="function", act="f32", weights="f32"),
        # One decode token of DeepSeek-V2-Lite: six experts, latency.
        _block("deepseek-bf16-1", "deepseek", 1),
        # A decode batch of Mixtral on the residual stream: every expert's weights read once.
        _block("mixtral-sublayer-bf16-16", "mixtral", 16, form="sublayer"),
        # A ragged decode batch over Qwen3's 128 experts, skewed routing.
        _block("qwen3-bf16-57", "qwen3", 57),
        # A chunk of a prompt beside running sequences, fp8 weights.
        _block("mixtral-fp8-333", "mixtral", 333, weights="fp8"),
        # A prompt on Qwen3's residual stream, a length that divides nothing.
        _block("qwen3-sublayer-bf16-2043", "qwen3", 2043, form="sublayer"),
        # Prefill with fp8 weights and two-term fp8 activations.
        _block("mixtral-fp8x2-3001", "mixtral", 3001, weights="fp8", fp8_act="x2"),
        # The largest prefill batch of the Mixtral configuration.
        _block("mixtral-bf16-4096", "mixtral", 4096),
        # The reference's type at a full model's size: a prompt in fp32.
        _block("deepseek-f32-500", "deepseek", 500, act="f32", weights="f32"),
        # The expert-selected product by itself, as a program that composes its own FFN calls it.
        _mmid("mul_mat_id-deepseek-up-bf16-96", "deepseek", "up", 96),
        # The decode step's attention sub-layer: 16 sequences of 4096 positions.
        _attention("attention-16x4096", "mixtral", 16, 4096, False, False),
        # A wide decode batch of shorter sequences of unequal length, with biases.
        _attention("attention-bias-61x1000", "mixtral", 61, 1000, True, True),
    ]


def _log_int(rng, lo, hi):
    return int(min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng):
    kind = rng.choices(["bf16", "fp8", "f32", "mul_mat_id", "attention"], [7, 4, 2, 3, 4])[0]
    if kind == "bf16":
        model = rng.choice(["mixtral", "qwen3", "deepseek"])
        c = _block("", model, _log_int(rng, 1, MAX_TOKENS[model]), form=rng.choice(["block", "sublayer"]))
    elif kind == "fp8":
        c = _block("", "mixtral", _log_int(rng, 1, MAX_TOKENS["mixtral"]), form=rng.choice(["block", "sublayer"]),
                   weights="fp8", fp8_act=rng.choice(["none", "x2", "e4m3"]))
    elif kind == "f32":
        model = rng.choice(["toy", "deepseek"])
        form = rng.choice(["function", "block", "sublayer"])
        c = _block("", model, _log_int(rng, 1, MAX_TOKENS_F32[model]), form=form, act="f32", weights="f32")
    elif kind == "mul_mat_id":
        model = rng.choice(["mixtral", "qwen3", "deepseek", "toy"])
        act = "f32" if model == "toy" else "bf16"
        c = _mmid("", model, rng.choice(["up", "down"]), _log_int(rng, 1, 2048), act=act)
    else:
        model = rng.choice(["mixtral", "mixtral", "small"])
        act = rng.choice(["bf16", "bf16", "f32"])
        batch = _log_int(rng, 1, 128)
        # at most the listed 16 x 4096 positions in all
        context = _log_int(rng, 1, min(8192, 65536 // batch))
        weights = rng.choice(["bf16", "fp8"]) if act == "bf16" else "f32"
        c = _attention("", model, batch, context, rng.random() < 0.7, rng.random() < 0.5, act=act, weights=weights,
                       block_size=rng.choice([16, 32, 64]))
    del c["name"]
    return c


# ---------------------------------------------------------------- inputs
def _normal(g, shape, std=1.0, mean=0.0):
    return torch.empty(shape, dtype=torch.float32, device="cuda").normal_(mean, std, generator=g)


def _generator(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(int(seed))
    return g


def _quantize(w, dim):
    """(e4m3 codes, fp32 scales) with one scale per output channel, absmax / 448 over `dim`."""
    scale = w.abs().amax(dim=dim).clamp_min(1e-12) / 448.0
    return (w / scale.unsqueeze(dim)).to(torch.float8_e4m3fn), scale


def _rms_norm64(x, w):
    x = x.double()
    return x / (x.square().mean(dim=1, keepdim=True) + EPS).sqrt() * w.double()


def _gap(x, wr, k):
    """Per row, the smallest gap between neighbours among its k + 1 largest router probabilities."""
    p = torch.softmax(x.double() @ wr.double().T, dim=1)
    p = p.topk(min(k + 1, p.shape[1]), dim=1).values
    return (p[:, :-1] - p[:, 1:]).amin(dim=1)


def _expert_weights(g, shape, weights):
    """One expert tensor [n_out, n_in, n_expert] ~ N(0, 0.02^2): a tensor, or fp8 (codes, scales)."""
    w = _normal(g, shape, 0.02)
    if weights == "fp8":
        return _quantize(w, 1)
    return w.to(TORCH[weights])


def _block_inputs(case, seed):
    """Token rows (or residual rows and norm weight), router and expert weights.  A row whose
    router probabilities nearly tie is drawn again, so that every summation order routes alike."""
    H, F, E, k, _, margin, zipf = MODELS[case["model"]]
    g = _generator(seed)
    dt = TORCH[case["act"]]
    wr = _normal(g, (E, H), 0.02)
    if zipf:  # channel 0 of every row is (near) 1 and carries a per-expert bias of -zipf * ln(rank)
        rank = torch.randperm(E, generator=g, device="cuda") + 1
        wr[:, 0] = -zipf * rank.float().log()
    wr = wr.to(dt)
    norm = None
    if case["form"] == "sublayer":
        norm = _normal(g, (H,), 0.1, 1.0)
        if zipf:
            norm[0] = 1.0
        norm = norm.to(dt)

    def rows(n):
        x = _normal(g, (n, H))
        if zipf:
            x[:, 0] = 1.0
        if norm is not None:
            scale = torch.empty((n, 1), device="cuda").uniform_(math.log(0.25), math.log(4.0), generator=g).exp()
            x = x * scale
        return x.to(dt)

    def near_tie(x):
        if norm is None:
            return _gap(x, wr, k) < margin
        xn = _rms_norm64(x, norm)
        return torch.minimum(_gap(xn, wr, k), _gap(xn.to(dt), wr, k)) < margin

    x = rows(case["tokens"])
    again = near_tie(x).nonzero().flatten()
    for _ in range(400):
        if again.numel() == 0:
            break
        fresh = rows(again.numel())
        x[again] = fresh
        again = again[near_tie(fresh)]
    else:
        raise RuntimeError("no rows that meet the router margin")
    up, gate, down = (_expert_weights(g, s, case["weights"]) for s in ((F, H, E), (F, H, E), (H, F, E)))
    return {"x": x, "norm": norm, "wr": wr, "up": up, "gate": gate, "down": down}


def _mmid_inputs(case, seed):
    H, F, E, k = MODELS[case["model"]][:4]
    n_out, n_in = (F, H) if case["proj"] == "up" else (H, F)
    g = _generator(seed)
    w = _expert_weights(g, (n_out, n_in, E), case["act"])
    x = _normal(g, (n_in, k, case["tokens"])).to(TORCH[case["act"]])
    ids = torch.rand((case["tokens"], E), generator=g, device="cuda").topk(k, dim=1).indices
    return {"w": w, "x": x, "ids": ids.T.to(torch.int32).contiguous()}


def _attention_inputs(case, seed):
    n_embd, n_head, n_kv = ATTENTION[case["model"]]
    D, B, bs, ctx = n_embd // n_head, case["batch"], case["block_size"], case["context"]
    g = _generator(seed)
    dt = TORCH[case["act"]]
    kv = n_kv * D
    shapes = ((n_embd, n_embd), (n_embd, kv), (n_embd, kv), (n_embd, n_embd))
    wdt = "bf16" if case["weights"] == "fp8" else case["weights"]
    w = [_normal(g, s, n_embd ** -0.5).to(TORCH[wdt]) for s in shapes]
    b = [_normal(g, (s[1],), 0.1) for s in shapes] if case["bias"] else [None] * 4
    lens = torch.full((B,), ctx, dtype=torch.int32, device="cuda")
    if case["ragged"]:
        lens = torch.randint(max(1, ctx // 2), ctx + 1, (B,), generator=g, device="cuda", dtype=torch.int32)
        lens[0] = ctx
    per_seq = ctx // bs + 1  # room for the new token
    order = torch.randperm(B * per_seq, generator=g, device="cuda").to(torch.int32)
    tables = order.view(1, B, per_seq).contiguous()
    pools = [_normal(g, (B * per_seq, bs, n_kv, D)).to(dt) for _ in range(2)]
    slot = torch.take_along_dim(tables[0], (lens // bs).long()[:, None], dim=1)[:, 0].contiguous()
    return {"x": _normal(g, (B, n_embd)).to(dt), "norm": _normal(g, (n_embd,), 0.1, 1.0).to(dt), "w": w, "b": b,
            "lens": lens, "tables": tables, "k": pools[0], "v": pools[1], "block": slot,
            "pos": (lens % bs).to(torch.int32).contiguous()}


# ---------------------------------------------------------------- the calls
def prepare(case, seed):
    if case["kind"] == "mul_mat_id":
        t = _mmid_inputs(case, seed)
        return {"kind": "mul_mat_id", "w": fm.pack_expert_weights(t["w"]), "x": t["x"], "ids": t["ids"]}
    if case["kind"] == "attention":
        t = _attention_inputs(case, seed)
        n_embd, n_head, n_kv = ATTENTION[case["model"]]
        attn = fm.AttentionBlockDecode(*t["w"], *t["b"], case["bias"], n_head=n_head, n_head_kv=n_kv, n_embd=n_embd,
                                       act_dtype=TORCH[case["act"]],
                                       weight_dtype="fp8" if case["weights"] == "fp8" else None)
        lens = t["lens"].view(1, -1).contiguous()
        args = (t["x"], t["norm"], EPS, t["lens"].long(), t["k"], t["v"], 0, t["tables"], lens, case["context"],
                t["block"], t["pos"])
        return {"kind": "attention", "attn": attn, "args": args}
    t = _block_inputs(case, seed)
    H, F, E, k, normalize = MODELS[case["model"]][:5]
    if case["form"] == "function":
        return {"kind": "function", "args": (t["x"], t["wr"], t["up"], t["gate"], t["down"], E, k, H, F, normalize)}
    weights = [fm.pack_expert_weights(fm.QuantizedExpertWeights(*t[n]) if case["weights"] == "fp8" else t[n])
               for n in ("up", "gate", "down")]
    fp8_act = {"none": False, "e4m3": True, "x2": "x2"}[case["fp8_act"]]
    block = fm.MoEFFNBlock(t["wr"], *weights, E, k, H, F, normalize, act_dtype=TORCH[case["act"]],
                           fp8_activations=fp8_act)
    return {"kind": case["form"], "block": block, "x": t["x"], "norm": t["norm"]}


def run(state):
    kind = state["kind"]
    if kind == "block":
        return state["block"](state["x"])
    if kind == "sublayer":
        return state["block"].sublayer(state["x"], state["norm"], EPS)
    if kind == "function":
        return fm.moe_ffn_block(*state["args"])
    if kind == "mul_mat_id":
        return fm.mul_mat_id(state["w"], state["x"], state["ids"])
    out, k_new, v_new = state["attn"].paged_sublayer(*state["args"])
    return {"out": out, "k_new": k_new, "v_new": v_new, "k_pool": state["args"][4], "v_pool": state["args"][5]}


# ---------------------------------------------------------------- what a call cannot do without
def _touched(E, k, tokens, zipf):
    """Expected number of experts that `tokens` tokens route to."""
    if not zipf:
        return E * (1.0 - (1.0 - k / E) ** tokens)
    p = [r ** -zipf for r in range(1, E + 1)]
    total = sum(p)
    return sum(1.0 - (1.0 - v / total) ** (k * tokens) for v in p)


def work(case):
    if case["kind"] == "attention":
        n_embd, n_head, n_kv = ATTENTION[case["model"]]
        B, kv, a = case["batch"], n_kv * (n_embd // n_head), BYTES[case["act"]]
        positions = B * case["context"] * (0.75 if case["ragged"] else 1.0)
        params = n_embd * (2 * n_embd + 2 * kv)
        return {"bytes": params * BYTES[case["weights"]] + 2 * positions * kv * a + B * (2 * n_embd + 4 * kv) * a,
                "flops": 2.0 * B * params + 4.0 * positions * n_embd}
    H, F, E, k, _, _, zipf = MODELS[case["model"]]
    T, a = case["tokens"], BYTES[case["act"]]
    if case["kind"] == "mul_mat_id":
        return {"bytes": _touched(E, k, T, 0.0) * H * F * a + T * k * ((H + F) * a + 4), "flops": 2.0 * T * k * H * F}
    return {"bytes": _touched(E, k, T, zipf) * 3 * H * F * BYTES[case["weights"]] + (E * H + 2 * T * H) * a,
            "flops": 2.0 * T * H * E + 6.0 * T * k * H * F}


def tolerance(case):
    """About four times the distance from ``exact`` that listed and drawn cases
    showed: 1.9e-6 in fp32; 3e-3 in bf16 (the SwiGLU rows, the weighted expert
    rows and the output are each rounded once), up to 0.06 of the RMS in one
    value; 0.047 with one e4m3 term per activation, 0.37 in one value."""
    if case["act"] == "f32":
        return {"rel": 8e-6, "max": 8e-5}
    if case["kind"] == "block":
        return {"rel": 1.9e-1, "max": 0.95} if case["fp8_act"] == "e4m3" else {"rel": 1.2e-2, "max": 0.25}
    return {"rel": 1.0e-2, "max": 0.04}


# ---------------------------------------------------------------- 64-bit results
def _full(w, e=None):
    """An expert tensor (of expert `e`, or a whole [n_in, n_out] matrix) in 64 bits, fp8 codes times their scales."""
    if isinstance(w, tuple):
        q, s = w
        return (q[:, :, e].double() * s[:, e].double()[:, None]) if e is not None else q.double() * s.double()
    return w[:, :, e].double() if e is not None else w.double()


def _exact_block(case, seed):
    t = _block_inputs(case, seed)
    _, _, E, k, normalize, _, _ = MODELS[case["model"]]
    x = t["x"].double() if t["norm"] is None else _rms_norm64(t["x"], t["norm"])
    p, ids = torch.softmax(x @ t["wr"].double().T, dim=1).topk(k, dim=1)
    if normalize:
        p = p / p.sum(dim=1, keepdim=True)
    out = torch.zeros_like(x) if t["norm"] is None else t["x"].double()
    for e in range(E):
        token, slot = (ids == e).nonzero(as_tuple=True)
        if token.numel() == 0:
            continue
        xe = x[token]
        up, gate = xe @ _full(t["up"], e).T.contiguous(), xe @ _full(t["gate"], e).T.contiguous()
        y = (gate * up * torch.sigmoid(up)) @ _full(t["down"], e).T.contiguous()
        out.index_add_(0, token, y * p[token, slot][:, None])
    return out


def _exact_mmid(case, seed):
    t = _mmid_inputs(case, seed)
    n_in, k, T = t["x"].shape
    x = t["x"].double().reshape(n_in, k * T).T.contiguous()
    flat = t["ids"].reshape(-1)
    out = torch.zeros((k * T, t["w"].shape[0]), dtype=torch.float64, device="cuda")
    for e in flat.unique().tolist():
        rows = (flat == e).nonzero().flatten()
        out[rows] = x[rows] @ _full(t["w"], e).T.contiguous()
    return out.T.contiguous().view(-1, k, T)


def _rope(x, positions):
    """Adjacent pairs (2i, 2i + 1) of x [B, heads, D] turned by position / 10000^(2i / D)."""
    D = x.shape[-1]
    i = torch.arange(D // 2, dtype=torch.float64, device=x.device)
    angle = positions.double()[:, None] / 10000.0 ** (2 * i / D)
    c, s = angle.cos()[:, None, :], angle.sin()[:, None, :]
    x0, x1 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x0 * c - x1 * s, x0 * s + x1 * c], dim=-1).flatten(-2)


def _exact_attention(case, seed):
    t = _attention_inputs(case, seed)
    n_embd, n_head, n_kv = ATTENTION[case["model"]]
    D, B, bs = n_embd // n_head, case["batch"], case["block_size"]
    w = [_full(_quantize(m.float(), 0)) if case["weights"] == "fp8" else m.double() for m in t["w"]]
    xn = _rms_norm64(t["x"], t["norm"])
    q, k, v = (xn @ m + (0.0 if b is None else b.double()) for m, b in zip(w[:3], t["b"][:3]))
    q = _rope(q.view(B, n_head, D), t["lens"])
    k = _rope(k.view(B, n_kv, D), t["lens"])
    v = v.view(B, n_kv, D)
    att = torch.empty((B, n_head, D), dtype=torch.float64, device="cuda")
    for s, n in enumerate(t["lens"].tolist()):
        blocks = t["tables"][0, s].long()
        kc, vc = (torch.cat([p[blocks].double().view(-1, n_kv, D)[:n], new[s][None]]).transpose(0, 1)
                  for p, new in ((t["k"], k), (t["v"], v)))
        qs = q[s].view(n_kv, n_head // n_kv, D)
        score = (qs @ kc.transpose(1, 2).contiguous()) * D ** -0.5
        # the positions from this sequence's length to the longest one's are keys and values of zeros
        top = score.amax(dim=-1, keepdim=True).clamp_min(0.0 if n < case["context"] else -math.inf)
        weight = (score - top).exp()
        total = weight.sum(dim=-1, keepdim=True) + (case["context"] - n) * (-top).exp()
        att[s] = (weight @ vc.contiguous() / total).view(n_head, D)
    out = att.view(B, n_embd) @ w[3] + (0.0 if t["b"][3] is None else t["b"][3].double()) + t["x"].double()
    pools = []
    for p, new in ((t["k"], k), (t["v"], v)):
        p = p.double()
        p[t["block"].long(), t["pos"].long()] = new
        pools.append(p)
    return {"out": out, "k_new": k, "v_new": v, "k_pool": pools[0], "v_pool": pools[1]}


def exact(case, seed):
    """What ``run`` returns on ``prepare(case, seed)``'s inputs, in 64 bits."""
    if case["kind"] == "mul_mat_id":
        return _exact_mmid(case, seed)
    if case["kind"] == "attention":
        return _exact_attention(case, seed)
    return _exact_block(case, seed)
