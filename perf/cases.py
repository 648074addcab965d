"""The work that a user of the dilution-attention library has it do, case by case.

    listed()             the named cases
    draw(rng)            one more case of the same ranges
    prepare(case, seed)  what a program holds before the call: inputs, caches, weights
    run(state)           one pass through the public entry points, with its outputs
    work(case)           bytes and operations that one pass cannot do without
    tolerance(case)      how far another correct implementation may be off
    exact(case, seed)    the outputs in float64, in plain torch

Kinds of cases:

    train    forward and backward of the operator (``kernels.dilution_attention``,
             or a bid variant through ``kernels_bid``).  layout "packed": q, k, v are
             views of one (B, T, 3 H D) projection and the output goes back to
             (B, T, H D) in the activations' type, as an attention layer calls it;
             "separate": contiguous (B, H, T, D) tensors, as a benchmark or an
             operator test calls it.
    forward  inference: the forward alone, no aux.
    prefill  a prompt into a decode cache (``cache.begin_cache``), in chunks.
    decode   one cached decode step for every sequence of a batch.
    lm       one decode step of a whole language model: logits from its caches.
"""

import math
import os
import sys

import torch

_PKG = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "dilution-attention_amd")
if _PKG not in sys.path:
    sys.path.insert(0, _PKG)

from dilution import cache as dcache  # noqa: E402
from dilution import kernels, kernels_bid  # noqa: E402
from dilution.lm import DilutionLM, LMConfig  # noqa: E402

DEV = "cuda"
EPS = 1e-9
VOCAB = 50304
_TYPES = {"bf16": torch.bfloat16, "fp32": torch.float32}


def _train(name, b, h, t, d, prec="bf16", layout="separate", bid="softmax"):
    return {"name": name, "kind": "train", "b": b, "h": h, "t": t, "d": d, "prec": prec, "layout": layout, "bid": bid}


def listed():
    return [
        # a short training call: the operator tests' shape (4 heads of 512 rows); launches and latency count
        _train("train_small", 1, 4, 512, 64),
        # an odd length, a head count that divides nothing, strided views of the layer's projection
        _train("train_ragged", 3, 5, 1357, 64, layout="packed"),
        # a training layer of the language model at a 2K context, as its attention layer calls the operator
        _train("train_2k", 8, 16, 2048, 64, layout="packed"),
        # the headline benchmark: one sequence of 16K
        _train("train_16k", 1, 16, 16384, 64),
        # heads of 128 at a 4K context
        _train("train_d128", 2, 8, 4096, 128),
        # fp32 activations: the precision that the model picks for them
        _train("train_tf32", 2, 8, 2048, 64, prec="tf32"),
        # a bid function of the ablation family
        _train("train_sigmoid", 2, 8, 4096, 64, bid="sigmoid"),
        # the bare forward in its default precision, fp32 operands
        {"name": "forward_ieee", "kind": "forward", "b": 1, "h": 4, "t": 512, "d": 64, "prec": "ieee"},
        # a batch of 8K prompts prefilled in the model's 2K chunks
        {"name": "prefill_8k", "kind": "prefill", "b": 4, "h": 16, "t": 8192, "d": 64, "prec": "bf16", "chunk": 2048},
        # one sequence's decode step at a short context: the smallest call
        {"name": "decode_short", "kind": "decode", "b": 1, "h": 16, "len": 1000, "d": 64, "prec": "bf16"},
        # serving 16 sequences at 128K
        {"name": "decode_128k", "kind": "decode", "b": 16, "h": 16, "len": 131072, "d": 64, "prec": "bf16"},
        # a token of 8 sequences through a 4-layer model at a 4K context
        {"name": "lm_token", "kind": "lm", "b": 8, "layers": 4, "d_model": 1024, "len": 4000},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _cost(c):
    """Score-sized work of a train / forward / prefill case, in bf16 head_dim-64 terms."""
    rate = {"bf16": 1.0, "tf32": 3.0, "ieee": 8.0}[c["prec"]] * (1.6 if c.get("bid", "softmax") != "softmax" else 1.0)
    products = 7 if c["kind"] == "train" else 2
    return products * rate * c["b"] * c["h"] * c["t"] ** 2 * max(c["d"], 64)


def draw(rng):
    kind = rng.choice(["train", "train", "train", "train", "forward", "prefill", "decode", "decode", "lm"])
    while True:
        b, h = _log_int(rng, 1, 16), rng.choice([1, 2, 3, 4, 5, 8, 12, 16])
        d = rng.choice([32, 64, 64, 64, 128])
        if kind == "lm":
            return {"kind": "lm", "b": rng.randint(1, 8), "layers": rng.randint(2, 4),
                    "d_model": rng.choice([512, 1024]), "len": _log_int(rng, 200, 8000)}
        if kind == "decode":
            c = {"kind": "decode", "b": b, "h": h, "len": _log_int(rng, 100, 131072), "d": d,
                 "prec": rng.choice(["bf16", "bf16", "bf16", "fp32"])}
            if work(c)["bytes"] <= 8.0e9:
                return c
            continue
        c = {"kind": kind, "b": b, "h": h, "t": _log_int(rng, 64, 16384), "d": d,
             "prec": rng.choice(["bf16", "bf16", "bf16", "bf16", "tf32"])}
        if kind == "train":
            c["layout"] = rng.choice(["packed", "separate"])
            c["bid"] = rng.choice(["softmax", "softmax", "softmax", "softmax", "sigmoid", "softplus"])
            if c["bid"] != "softmax":
                c["prec"] = "bf16"
        elif kind == "forward":
            c["prec"] = rng.choice(["bf16", "tf32", "ieee"])
        else:
            c["t"] = min(c["t"], 8192)
            chunk = rng.choice([512, 1024, 2048, _log_int(rng, 100, 3000)])
            c["chunk"] = max(chunk, c["t"] // 16)
        if _cost(c) <= 1.9e12:
            return c


# ---------------------------------------------------------------------------
# inputs


def _gen(seed):
    g = torch.Generator(device=DEV)
    g.manual_seed(seed)
    return g


def _randn(g, shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=g, device=DEV, dtype=torch.float32) * scale).to(dtype)


def _dtype(case):
    return torch.bfloat16 if case["prec"] == "bf16" else torch.float32


def _operator_inputs(case, seed):
    """q, k ~ 0.5 N(0, 1), v and dout ~ N(0, 1) (the benchmark's distribution)."""
    g, dt = _gen(seed), _dtype(case)
    b, h, t, d = case["b"], case["h"], case["t"], case["d"]
    if case.get("layout") == "packed":
        qkv = torch.cat([_randn(g, (b, t, h * d), dt, s) for s in (0.5, 0.5, 1.0)], dim=2)
        return qkv, _randn(g, (b, t, h * d), dt)
    shape = (b, h, t, d)
    return [_randn(g, shape, dt, s) for s in (0.5, 0.5, 1.0)], _randn(g, shape, torch.float32)


def _split(qkv, h, d):
    """(B, H, T, D) views of a (B, T, 3 H D) projection, as the attention layer takes them."""
    b, t, _ = qkv.shape
    return [x.view(b, t, h, d).transpose(1, 2) for x in qkv.split(h * d, dim=2)]


def _demand(g, b, h, length, capacity):
    """A demand vector like the one a prefix of length - 1 rows leaves: early keys hold more; zero from the new row on."""
    pos = torch.arange(length - 1, device=DEV, dtype=torch.float32)
    com = torch.zeros(b, h, capacity, device=DEV)
    noise = torch.randn(b, h, length - 1, generator=g, device=DEV) * 0.5
    com[:, :, : length - 1] = torch.log(length / (pos + 1.0)) * torch.exp(noise)
    return com


def _decode_inputs(case, seed):
    g, dt = _gen(seed), _TYPES[case["prec"]]
    b, h, n, d = case["b"], case["h"], case["len"], case["d"]
    k, v = _randn(g, (b, h, n, d), dt), _randn(g, (b, h, n, d), dt)
    return _randn(g, (b, h, 1, d), dt), k, v, _demand(g, b, h, n, n)


def _lm_inputs(case, seed):
    """A randomly initialised bf16 model and caches holding `len` positions, with room for more."""
    torch.manual_seed(seed)
    cfg = LMConfig(vocab_size=VOCAB, n_layers=case["layers"], d_model=case["d_model"], n_heads=case["d_model"] // 64)
    with torch.device(DEV):
        model = DilutionLM(cfg).to(torch.bfloat16).eval()
    g = _gen(seed)
    b, h, n = case["b"], cfg.n_heads, case["len"]
    caches = []
    for _ in range(cfg.n_layers):
        shape = (b, h, n + 64, 64)
        caches.append({"k": _randn(g, shape, torch.bfloat16, 0.6), "v": _randn(g, shape, torch.bfloat16, 0.6), "len": n,
                       "committed": _demand(g, b, h, n + 1, n + 64)})
    return model, torch.randint(0, VOCAB, (b, 1), generator=g, device=DEV), caches


def prepare(case, seed):
    state = {"case": case}
    if case["kind"] in ("train", "forward", "prefill"):
        x, dout = _operator_inputs(case, seed)
        if case["kind"] == "train":
            state["leaves"] = [t.requires_grad_(True) for t in (x if isinstance(x, list) else [x])]
            state["dout"] = dout
        else:
            state["qkv"] = x
    elif case["kind"] == "decode":
        state["q1"], state["k"], state["v"], state["committed"] = _decode_inputs(case, seed)
    else:
        state["model"], state["token"], state["caches"] = _lm_inputs(case, seed)
    return state


# ---------------------------------------------------------------------------
# one pass


def _run_train(state):
    case, leaves = state["case"], state["leaves"]
    h, d = case["h"], case["d"]
    packed = case["layout"] == "packed"
    q, k, v = _split(leaves[0], h, d) if packed else leaves
    if case["bid"] == "softmax":
        out = kernels.dilution_attention(q, k, v, dot_precision=case["prec"])
    else:
        out = kernels_bid.dilution_attention(q, k, v, dot_precision=case["prec"], bid=case["bid"])
    if packed:
        out = out.to(q.dtype).transpose(1, 2).contiguous().view(case["b"], case["t"], h * d)
        grads = torch.autograd.grad(out, leaves, state["dout"])
        return {"out": out.detach(), "dqkv": grads[0]}
    dq, dk, dv = torch.autograd.grad(out, leaves, state["dout"])
    return {"out": out.detach(), "dq": dq, "dk": dk, "dv": dv}


def run(state):
    case = state["case"]
    if case["kind"] == "train":
        return _run_train(state)
    with torch.no_grad():
        if case["kind"] == "forward":
            q, k, v = state["qkv"]
            return {"out": kernels.dilution_attention_forward(q, k, v, dot_precision=case["prec"])}
        if case["kind"] == "prefill":
            q, k, v = state["qkv"]
            y, cache = dcache.begin_cache(q, k, v, chunk=case["chunk"], dot_precision=case["prec"])
            return {"y": y, "k": cache["k"], "v": cache["v"], "committed": cache["committed"]}
        if case["kind"] == "decode":
            y = kernels.dilution_decode_step(state["q1"], state["k"], state["v"], state["committed"], case["len"])
            return {"y": y, "committed": state["committed"]}
        # the same position each time: the caches' length is the caller's
        caches = [dict(c, len=case["len"]) for c in state["caches"]]
        logits = state["model"].decode_step(state["token"], caches)
        return {"logits": logits, "committed": [c["committed"] for c in caches]}


# ---------------------------------------------------------------------------
# what a pass cannot do without


def work(case):
    if case["kind"] == "lm":
        dm, layers, n = case["d_model"], case["layers"], case["len"] + 1
        weights = layers * (4 * dm * dm + 3 * 4 * dm * dm) + VOCAB * dm
        cached = layers * case["b"] * dm * n
        return {"bytes": 2 * weights + cached * 4 + cached // 64 * 8 + 2 * case["b"] * VOCAB,
                "flops": 2 * case["b"] * weights + 4 * cached}
    size = 2 if case["prec"] == "bf16" else 4
    n, d = case["b"] * case["h"], case["d"]
    if case["kind"] == "decode":
        return {"bytes": n * case["len"] * (2 * d * size + 8), "flops": 4 * n * case["len"] * d}
    t = case["t"]
    rows = n * t * d
    if case["kind"] == "train":
        ends = size if case["layout"] == "packed" else 4          # the output and its gradient
        return {"bytes": rows * (6 * size + 2 * ends), "flops": 7 * n * t * t * d}
    if case["kind"] == "forward":
        return {"bytes": rows * (3 * size + 4), "flops": 2 * n * t * t * d}
    return {"bytes": rows * 6 * size + n * t * 4, "flops": 2 * n * t * t * d}


# ---------------------------------------------------------------------------
# how far off


def tolerance(case):
    # about four times the distance from exact() that these paths show over the
    # declared ranges: bf16 operands (2^-9 each) in every product; tf32: split
    # operands of about 16 bits; ieee and fp32 decode: fp32 sums.  A model's
    # logits carry the roundings of all its layers.
    if case["kind"] == "lm":
        return {"rel": 5e-2, "max": 0.25}
    if case["kind"] == "decode":
        return {"rel": 7e-3, "max": 1.6e-2} if case["prec"] == "bf16" else {"rel": 1.5e-6, "max": 1e-5}
    return {"bf16": {"rel": 1.4e-2, "max": 0.25}, "tf32": {"rel": 3e-5, "max": 4e-4},
            "ieee": {"rel": 1e-6, "max": 1e-5}}[case["prec"]]


# ---------------------------------------------------------------------------
# the same in float64


def _weights64(q, k, bid="softmax"):
    """The attention weights of one slice and the column totals of its bids."""
    t, d = q.shape
    a = (q @ k.T) / math.sqrt(d)
    causal = torch.ones(t, t, dtype=torch.bool, device=q.device).tril()
    if bid == "softmax":
        p = torch.softmax(a.masked_fill(~causal, float("-inf")), dim=1)
    elif bid == "sigmoid":
        p = torch.sigmoid(a).masked_fill(~causal, 0.0)
    else:
        p = torch.nn.functional.softplus(a).masked_fill(~causal, 0.0)
        p = p / p.sum(dim=1, keepdim=True)
    total = p.cumsum(dim=0)
    share = p / (total + EPS)                                     # demand of the earlier rows + p + eps
    return share / (share.sum(dim=1, keepdim=True) + EPS), total[-1]


def _exact_operator(case, seed):
    x, dout = _operator_inputs(case, seed)
    b, h, t, d = case["b"], case["h"], case["t"], case["d"]
    packed = case.get("layout") == "packed"
    qkv = _split(x, h, d) if packed else x
    back = case["kind"] == "train"
    if back:
        dout = dout.view(b, t, h, d).transpose(1, 2) if packed else dout
    f64 = dict(device=DEV, dtype=torch.float64)
    got = [torch.empty(b, h, t, d, **f64) for _ in range(4 if back else 1)]
    total = torch.empty(b, h, t, **f64)
    for i in range(b):
        for j in range(h):
            xs = [y[i, j].detach().double().requires_grad_(back) for y in qkv]
            w, tot = _weights64(xs[0], xs[1], case.get("bid", "softmax"))
            out = w @ xs[2]
            parts = [out.detach()]
            total[i, j] = tot.detach()
            if back:
                parts += torch.autograd.grad(out, xs, dout[i, j].double())
            del w, out
            for g, p in zip(got, parts):
                g[i, j] = p
    if case["kind"] == "forward":
        return {"out": got[0]}
    if case["kind"] == "prefill":
        return {"y": got[0], "k": qkv[1].double(), "v": qkv[2].double(), "committed": total}
    if packed:
        rows = [g.transpose(1, 2).reshape(b, t, h * d) for g in got]
        return {"out": rows[0], "dqkv": torch.cat(rows[1:], dim=2)}
    return dict(zip(("out", "dq", "dk", "dv"), got))


def _decode64(q1, k, v, committed):
    """One step over whole caches: q1 (n, d), k and v (n, L, d), committed (n, L)."""
    a = torch.stack([k[i] @ q1[i] for i in range(k.shape[0])]) / math.sqrt(q1.shape[1])
    p = torch.softmax(a, dim=1)
    share = p / (committed + p + EPS)
    w = share / (share.sum(dim=1, keepdim=True) + EPS)
    return torch.stack([w[i] @ v[i] for i in range(k.shape[0])]), committed + p


def _exact_decode(case, seed):
    q1, k, v, com = _decode_inputs(case, seed)
    y = torch.empty(q1.shape, device=DEV, dtype=torch.float64)
    new = torch.empty(com.shape, device=DEV, dtype=torch.float64)
    for i in range(case["b"]):
        yi, ci = _decode64(q1[i, :, 0].double(), k[i].double(), v[i].double(), com[i].double())
        y[i, :, 0], new[i] = yi, ci
    return {"y": y, "committed": new}


def _exact_lm(case, seed):
    model, token, caches = _lm_inputs(case, seed)
    b, n, heads = case["b"], case["len"], model.cfg.n_heads

    def norm(x, m):
        return x * torch.rsqrt(x.square().mean(dim=-1, keepdim=True) + m.eps) * m.weight.detach().double()

    def lin(x, m):
        return x @ m.weight.detach().double().T

    x = model.wte.weight.detach()[token[:, 0]].double()
    news = []
    for block, c in zip(model.h, caches):
        q, k1, v1 = lin(norm(x, block.ln_1), block.attn.c_attn).split(model.cfg.d_model, dim=1)
        y = torch.empty_like(x).view(b, heads, 64)
        new = c["committed"].double()
        for i in range(b):
            k = torch.cat([c["k"][i, :, :n].double(), k1[i].view(heads, 1, 64)], dim=1)
            v = torch.cat([c["v"][i, :, :n].double(), v1[i].view(heads, 1, 64)], dim=1)
            y[i], new[i, :, : n + 1] = _decode64(q[i].view(heads, 64), k, v, new[i, :, : n + 1])
        news.append(new)
        x = x + lin(y.view(b, -1), block.attn.c_proj)
        r = norm(x, block.ln_2)
        x = x + lin(torch.nn.functional.silu(lin(r, block.mlp.gate_proj)) * lin(r, block.mlp.up_proj), block.mlp.down_proj)
    return {"logits": lin(norm(x, model.ln_f), model.lm_head).view(b, 1, -1), "committed": news}


def exact(case, seed):
    if case["kind"] == "decode":
        return _exact_decode(case, seed)
    if case["kind"] == "lm":
        return _exact_lm(case, seed)
    return _exact_operator(case, seed)
