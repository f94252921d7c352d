"""The work a program gives this framework, as cases that can be timed.

Everything goes through the public entry points: torch ops on "spyre"
tensors, torch.compile on them, HIP graphs (torch_spyre.graphs) and the
decoder of torch_spyre.examples.  The framework's ops are forward ops (it
registers no norm, softmax or attention gradients), so the directions are
prefill and decode.  Sizes are those of the repository's own workloads
(512 x 4096 softmax, 4096^3 product, 32 x 2048 x 2048 x 128 batched product,
8192 x 4096 row kernels, a 4096-wide decoder of 32 query and 8 key-value
heads with 12800-wide MLP and a vocabulary of 49155) and what a server does
around them: prompts of any length, decode batches from 1 to 32.
"""

import math
import os
import sys

import torch
import torch.nn.functional as F

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "torch-spyre_amd"))

import torch_spyre  # noqa: E402,F401  (registers the device)
import torch_spyre.graphs as graphs  # noqa: E402
from torch_spyre.examples import decoder as D  # noqa: E402

# One compiled graph per shape: a program that meets many shapes raises
# dynamo's limit of graphs per function.
torch._dynamo.config.recompile_limit = 256
torch._dynamo.config.accumulated_recompile_limit = 1024
torch._dynamo.config.fail_on_recompile_limit_hit = True

DTYPES = {"fp16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-5
HIDDEN, MLP, VOCAB = 4096, 12800, 49155
QKV = 6144


def listed():
    return [
        # one softmax call of attention-sized rows: the smallest eager call,
        # launch latency counts
        {"name": "softmax_1024x4096", "kind": "softmax", "rows": 1024, "cols": 4096,
         "log": False, "dtype": "fp16"},
        # token log-probabilities of a batch of 64 sequences: odd row length
        {"name": "log_softmax_64x49155", "kind": "softmax", "rows": 64, "cols": VOCAB, "log": True,
         "dtype": "bf16"},
        # residual add + RMSNorm between two sublayers, compiled
        {"name": "add_rmsnorm_8192x4096", "kind": "rows", "op": "rms", "rows": 8192,
         "cols": HIDDEN, "dtype": "fp16"},
        # fused pointwise chain with a row sum, compiled
        {"name": "gelu_rowsum_8192x4096", "kind": "rows", "op": "gelu", "rows": 8192,
         "cols": HIDDEN, "dtype": "bf16"},
        # down projection of a decode batch of 48 sequences
        {"name": "linear_48x4096x12800", "kind": "linear", "m": 48, "n": HIDDEN, "k": MLP,
         "bias": False, "dtype": "bf16"},
        # QKV projection (with bias) of one prompt of ordinary, odd length
        {"name": "linear_333x6144x4096", "kind": "linear", "m": 333, "n": QKV, "k": HIDDEN,
         "bias": True, "dtype": "fp16"},
        # large square product, both operands row-major
        {"name": "mm_4096", "kind": "mm", "m": 4096, "n": 4096, "k": 4096, "dtype": "fp16"},
        # attention-score-shaped batched product
        {"name": "bmm_32x2048x2048x128", "kind": "bmm", "batch": 32, "m": 2048, "n": 2048,
         "k": 128, "dtype": "fp16"},
        # one decoder layer over a full-length prompt, compiled
        {"name": "layer_1x2048", "kind": "layer", "batch": 1, "seq": 2048, "dtype": "fp16"},
        # prefill of three prompts of odd length into the KV cache, compiled
        {"name": "prefill_3x777", "kind": "prefill", "batch": 3, "seq": 777, "layers": 1,
         "dtype": "bf16"},
        # one decode step of a small batch, compiled and graph-replayed
        {"name": "decode_4_at_1100", "kind": "decode", "batch": 4, "pos": 1100, "max_len": 1152,
         "layers": 2, "dtype": "fp16"},
        # the same step at a serving batch
        {"name": "decode_24_at_700", "kind": "decode", "batch": 24, "pos": 700, "max_len": 1000,
         "layers": 2, "dtype": "bf16"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["softmax", "rows", "linear", "linear", "mm", "bmm", "layer", "prefill",
                       "decode", "decode"])
    c = {"kind": kind, "dtype": rng.choice(["fp16", "bf16"])}
    if kind == "softmax":
        cols = _log_int(rng, 64, 65536)
        c.update(rows=_log_int(rng, (1 << 22) // cols, (1 << 25) // cols), cols=cols,
                 log=rng.random() < 0.5)
    elif kind == "rows":
        cols = _log_int(rng, 256, 8192)
        if rng.random() < 0.75:
            cols = cols // 8 * 8
        c.update(op=rng.choice(["rms", "layer", "gelu"]),
                 rows=_log_int(rng, 1, min(16384, (1 << 25) // cols)), cols=cols)
    elif kind == "linear":
        m, n, k = _log_int(rng, 1, 4096), _log_int(rng, 256, VOCAB), _log_int(rng, 256, MLP)
        if rng.random() < 0.6:  # a model's own projection
            n, k = rng.choice([(QKV, HIDDEN), (HIDDEN, HIDDEN), (2 * MLP, HIDDEN), (HIDDEN, MLP),
                               (VOCAB, HIDDEN)])
        elif rng.random() < 0.75:
            k = k // 8 * 8
        m = max(1, min(m, (1 << 37) // (n * k)))
        c.update(m=m, n=n, k=k, bias=rng.random() < 0.5)
    elif kind == "mm":
        c.update(m=_log_int(rng, 128, 4096), n=_log_int(rng, 128, 4096), k=_log_int(rng, 128, 4096))
    elif kind == "bmm":
        m, n = _log_int(rng, 64, 2048), _log_int(rng, 64, 2048)
        c.update(batch=_log_int(rng, 2, 32), m=m, n=n,
                 k=rng.choice([64, 128, _log_int(rng, 32, 512)]))
    elif kind == "layer":
        c.update(batch=1, seq=_log_int(rng, 16, 2048))
    elif kind == "prefill":
        b = rng.randint(1, 4)
        c.update(batch=b, seq=_log_int(rng, 16, min(1024, 2331 // b)), layers=1)
    else:
        pos = _log_int(rng, 16, 1500)
        c.update(batch=_log_int(rng, 1, 24), pos=pos, max_len=pos + rng.randint(1, 200), layers=2)
    return c


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed))


def _config(case):
    return D.DecoderConfig(n_layers=case.get("layers", 1))


def _weights(g, cfg, dt):
    def normal(*shape, std=0.02, mean=0.0):
        return (torch.randn(*shape, generator=g, device="cuda") * std + mean).to(dt)

    h, kv = cfg.hidden, cfg.n_kv_heads * cfg.head_dim
    layers = [{"attn_norm": normal(h, mean=1.0), "wqkv": normal(h + 2 * kv, h),
               "wo": normal(h, h), "mlp_norm": normal(h, mean=1.0),
               "wgu": normal(2 * cfg.intermediate, h), "wd": normal(h, cfg.intermediate)}
              for _ in range(cfg.n_layers)]
    return {"embed": normal(cfg.vocab, h), "layers": layers}, normal


def _inputs(case, seed):
    """The case's inputs on the GPU as torch tensors of its type, from the
    seed alone."""
    g, dt, kind = _generator(seed), DTYPES[case["dtype"]], case["kind"]

    def normal(*shape, std=1.0, mean=0.0):
        return (torch.randn(*shape, generator=g, device="cuda") * std + mean).to(dt)

    if kind == "softmax":
        return {"x": normal(case["rows"], case["cols"], std=4.0)}
    if kind == "rows":
        c = case["cols"]
        return {"x": normal(case["rows"], c), "r": normal(case["rows"], c),
                "w": normal(c, std=0.1, mean=1.0), "b": normal(c, std=0.1)}
    if kind == "linear":
        d = {"x": normal(case["m"], case["k"]), "w": normal(case["n"], case["k"], std=0.02)}
        if case["bias"]:
            d["b"] = normal(case["n"], std=0.1)
        return d
    if kind == "mm":
        return {"a": normal(case["m"], case["k"]), "b": normal(case["k"], case["n"])}
    if kind == "bmm":
        return {"a": normal(case["batch"], case["m"], case["k"]),
                "b": normal(case["batch"], case["k"], case["n"])}
    cfg = _config(case)
    params, draw_weight = _weights(g, cfg, dt)
    d = {"params": params}
    if kind != "layer":
        params["final_norm"] = draw_weight(cfg.hidden, mean=1.0)
        params["lm_head"] = draw_weight(cfg.vocab, cfg.hidden)
    shape = (case["batch"],) if kind == "decode" else (case["batch"], case["seq"])
    d["tokens"] = torch.randint(0, cfg.vocab, shape, generator=g, device="cuda")
    if kind == "decode":
        cache = []
        for _ in range(cfg.n_layers):
            k = normal(case["batch"], cfg.n_kv_heads, case["max_len"], cfg.head_dim)
            v = normal(case["batch"], cfg.n_kv_heads, cfg.head_dim, case["max_len"])
            k[:, :, case["pos"]:] = 0
            v[:, :, :, case["pos"]:] = 0
            cache.append((k, v))
        d["cache"] = cache
    return d


def _move(v, where):
    if isinstance(v, torch.Tensor):
        return v.cpu().to(where)
    if isinstance(v, dict):
        return {k: _move(x, where) for k, x in v.items()}
    return [_move(x, where) for x in v] if isinstance(v, list) else \
        tuple(_move(x, where) for x in v)


def _add_rms(x, r, w, b):
    h = x + r
    return h, torch.rms_norm(h, [h.shape[-1]], w, EPS)


def _add_layer(x, r, w, b):
    h = x + r
    return h, F.layer_norm(h, [h.shape[-1]], w, b, EPS)


def _gelu_rowsum(x, r, w, b):
    y = F.gelu(x * w + b)
    return y, y.sum(-1)


_compiled = {f: torch.compile(f, dynamic=False) for f in
             (_add_rms, _add_layer, _gelu_rowsum, D.block_forward, D.layer_forward,
              D.decode_step_static)}
_ROWS = {"rms": _add_rms, "layer": _add_layer, "gelu": _gelu_rowsum}


def prepare(case, seed):
    kind, dt, dev = case["kind"], DTYPES[case["dtype"]], "spyre"
    s = _move(_inputs(case, seed), dev)
    s["kind"] = kind
    if kind == "softmax":
        s["fn"] = torch.log_softmax if case["log"] else torch.softmax
    elif kind == "rows":
        s["fn"] = _compiled[_ROWS[case["op"]]]
    elif kind in ("layer", "prefill", "decode"):
        s["cfg"] = cfg = _config(case)
        length = case["max_len"] if kind == "decode" else case["seq"]
        s["cos"], s["sin"] = D.rope_tables(cfg, length, dev, dt)
        if kind != "decode":
            s["mask"] = D.causal_mask(cfg, length, dev, dt)
        if kind == "layer":
            s["fn"] = _compiled[D.block_forward]
        if kind == "prefill":
            s["fn"] = _compiled[D.layer_forward]
            s["cache"] = D.new_cache(cfg, case["batch"], length, dev, dt)
        if kind == "decode":
            s["pos"] = torch.full((1,), case["pos"], dtype=torch.int64).to(dev)
            step = _compiled[D.decode_step_static]
            a = (s["tokens"], s["pos"], s["params"], s["cos"], s["sin"], s["cache"], cfg)
            step(*a)  # loads every kernel; writes what each replay writes
            s["graph"] = graphs.SpyreGraph()
            with graphs.graph(s["graph"]):
                s["logits"] = step(*a)
    return s


def run(s):
    kind = s["kind"]
    if kind == "softmax":
        return s["fn"](s["x"], -1)
    if kind == "rows":
        return s["fn"](s["x"], s["r"], s["w"], s["b"])
    if kind == "linear":
        return F.linear(s["x"], s["w"], s.get("b"))
    if kind == "mm":
        return s["a"] @ s["b"]
    if kind == "bmm":
        return torch.bmm(s["a"], s["b"])
    if kind == "layer":
        return s["fn"](s["tokens"], s["params"], s["cos"], s["sin"], s["mask"], s["cfg"])
    if kind == "prefill":
        logits = D.prefill(s["tokens"], s["params"], s["cos"], s["sin"], s["mask"], s["cache"],
                           s["cfg"], s["fn"])
    else:
        s["graph"].replay()
        logits = s["logits"]
    return {"logits": logits, "cache": s["cache"]}


def work(case):
    kind, e = case["kind"], 2
    if kind == "softmax":
        return {"bytes": 2 * e * case["rows"] * case["cols"], "flops": 0}
    if kind == "rows":
        r, c = case["rows"], case["cols"]
        if case["op"] == "gelu":  # reads x, w, b; writes y and the row sums
            return {"bytes": e * (2 * r * c + 2 * c + r), "flops": 0}
        return {"bytes": e * (4 * r * c + (2 if case["op"] == "layer" else 1) * c), "flops": 0}
    if kind in ("linear", "mm", "bmm"):
        bs, m, n, k = case.get("batch", 1), case["m"], case["n"], case["k"]
        return {"bytes": e * (bs * (m * k + n * k + m * n) + (n if case.get("bias") else 0)),
                "flops": 2 * bs * m * n * k}
    cfg = _config(case)
    h, d = cfg.hidden, cfg.head_dim
    per_layer = h * (h + 2 * cfg.n_kv_heads * d) + h * h + 3 * h * cfg.intermediate
    b = case["batch"]
    t = b if kind == "decode" else b * case["seq"]
    # keys that a query sees: all of them up to its own position
    seen = (case["pos"] + 1) * b if kind == "decode" else b * case["seq"] * (case["seq"] + 1) // 2
    flops = cfg.n_layers * (2 * t * per_layer + 4 * seen * cfg.n_heads * d)
    kv = 2 * cfg.n_kv_heads * d * (seen if kind == "decode" else t)
    byts = e * (cfg.n_layers * (per_layer + 2 * h) + t * h)  # weights, embedding rows
    if kind == "layer":
        return {"bytes": byts + e * t * h, "flops": flops}
    head = cfg.vocab * h
    return {"bytes": byts + e * (cfg.n_layers * kv + head + h + b * cfg.vocab),
            "flops": flops + 2 * b * head}


def tolerance(case):
    fp16 = case["dtype"] == "fp16"
    if case["kind"] in ("layer", "prefill", "decode"):
        return {"rel": 5e-3 if fp16 else 3e-2, "max": 4e-2 if fp16 else 2.5e-1}
    return {"rel": 1e-3 if fp16 else 8e-3, "max": 8e-3 if fp16 else 6e-2}


def _layer64(h, w, cfg, cos, sin, see, old=None):
    """One decoder layer on h [B, S, hidden] in 64 bits: (output, K
    [B, 8, S, D], V).  `see` [S, keys] says which key a query sees; `old`
    holds the cached K, V [B, 8, P, D] in front of the new ones."""
    B, S, H = h.shape
    d, kvh, g = cfg.head_dim, cfg.n_kv_heads, cfg.group

    def norm(t, weight):
        return t * torch.rsqrt(t.square().mean(-1, keepdim=True) + cfg.eps) * weight

    def rope(t):  # [B, heads, S, D]
        half = d // 2
        return t * cos + torch.cat([-t[..., half:], t[..., :half]], -1) * sin

    qkv = norm(h, w["attn_norm"].double()).reshape(B * S, H) @ w["wqkv"].double().t().contiguous()
    q, k, v = qkv.split([H, kvh * d, kvh * d], -1)
    q = rope(q.reshape(B, S, -1, d).transpose(1, 2))
    k = rope(k.reshape(B, S, kvh, d).transpose(1, 2))
    v = v.reshape(B, S, kvh, d).transpose(1, 2)
    keys, vals = (k, v) if old is None else (torch.cat([o, t], 2) for o, t in zip(old, (k, v)))
    o = torch.empty_like(q)
    for i in range(q.shape[1]):
        s = torch.bmm(q[:, i], keys[:, i // g].transpose(1, 2).contiguous()) / math.sqrt(d)
        p = torch.softmax(s.masked_fill(~see, float("-inf")), -1)
        o[:, i] = torch.bmm(p, vals[:, i // g].contiguous())
    h = h + (o.transpose(1, 2).reshape(B * S, H) @ w["wo"].double().t().contiguous()).view(B, S, H)
    gu = norm(h, w["mlp_norm"].double()).reshape(B * S, H) @ w["wgu"].double().t().contiguous()
    a = F.silu(gu[:, :cfg.intermediate]) * gu[:, cfg.intermediate:]
    return h + (a @ w["wd"].double().t().contiguous()).view(B, S, H), k, v


def exact(case, seed):
    kind = case["kind"]
    d = _inputs(case, seed)
    if kind == "softmax":
        return (torch.log_softmax if case["log"] else torch.softmax)(d["x"].double(), -1)
    if kind == "rows":
        x, r, w, b = (d[n].double() for n in ("x", "r", "w", "b"))
        if case["op"] == "gelu":
            y = F.gelu(x * w + b)
            return y, y.sum(-1)
        h = x + r
        if case["op"] == "layer":
            return h, F.layer_norm(h, [h.shape[-1]], w, b, EPS)
        return h, h * torch.rsqrt(h.square().mean(-1, keepdim=True) + EPS) * w
    if kind == "linear":
        y = d["x"].double() @ d["w"].double().t().contiguous()
        return y + d["b"].double() if "b" in d else y
    if kind == "mm":
        return d["a"].double() @ d["b"].double()
    if kind == "bmm":
        return torch.bmm(d["a"].double(), d["b"].double())
    cfg, dt, p = _config(case), DTYPES[case["dtype"]], d["params"]
    step = kind == "decode"
    length = case["max_len"] if step else case["seq"]
    cos, sin = (t.double() for t in D.rope_tables(cfg, length, "cuda", dt))
    h = p["embed"][d["tokens"]].double()
    if step:
        at = case["pos"]
        h, cos, sin = h[:, None], cos[at:at + 1], sin[at:at + 1]
        see = torch.ones(1, at + 1, dtype=torch.bool, device="cuda")
    else:
        see = torch.ones(length, length, dtype=torch.bool, device="cuda").tril()
    cache = []
    for i, w in enumerate(p["layers"]):
        if step:
            kc, vc = (t.double() for t in d["cache"][i])
            h, k, v = _layer64(h, w, cfg, cos, sin, see,
                               (kc[:, :, :at], vc[..., :at].transpose(2, 3)))
            kc[:, :, at:at + 1], vc[..., at:at + 1] = k, v.transpose(2, 3)
            cache.append((kc, vc))
        else:
            h, k, v = _layer64(h, w, cfg, cos, sin, see)
            cache.append((k, v.transpose(2, 3).contiguous()))
    if kind == "layer":
        return h
    x = h[:, -1]
    x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + cfg.eps) * p["final_norm"].double()
    return {"logits": x @ p["lm_head"].double().t().contiguous(), "cache": cache}
