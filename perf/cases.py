"""Timing cases of the library: what a program has it do, through its public
entry points (`tessel_amd.kernel` / `launch`, and `Engine`), from one-token
calls to the largest, with ragged and odd sizes among them.

A case is a dict of plain values; `kind` says which of the families below it
belongs to. `prepare` makes its inputs on the GPU, `run` is one pass,
`exact` the same outputs in 64 bits by plain torch.
"""

import math

import numpy as np
import torch

import tessel_amd as T

DEV = "cuda"

# Decoder shapes of the repository's configurations (dim, ffn): TinyLlama's,
# the ones its tests use at 1024 and 4096 columns, and the tiny model's.
BLOCKS = ((2048, 5632), (1024, 4000), (4096, 11008), (64, 128))


def listed():
    return [
        # A decoder MLP for one token: a single chat session, four launches.
        {"name": "mlp_1_token", "kind": "mlp", "rows": 1, "dim": 2048, "ffn": 5632},
        # The same for a short prompt of odd length: between decode and full prefill.
        {"name": "mlp_213_tokens", "kind": "mlp", "rows": 213, "dim": 2048, "ffn": 5632},
        # Final norm and output projection for a full decode batch beyond 32 rows.
        {"name": "head_48_rows", "kind": "head", "rows": 48, "tokens": 48, "dim": 2048, "vocab": 32000},
        # A matrix product nobody padded: every dimension odd.
        {"name": "matmul_odd", "kind": "matmul", "op": "matmul", "m": 777, "n": 1155, "k": 1001},
        # The headline product.
        {"name": "matmul_4096", "kind": "matmul", "op": "matmul", "m": 4096, "n": 4096, "k": 4096},
        # The single-precision product.
        {"name": "matmul_f32_1024", "kind": "matmul", "op": "matmul_f32", "m": 1024, "n": 1024, "k": 1024},
        # Causal attention at the benchmark's longest sequence.
        {"name": "flash_4096", "kind": "attention", "op": "flash", "heads": 32, "kv_heads": 32, "dim": 64, "seq": 4096,
         "prompts": 1},
        # Wider heads and a sequence that no tile divides.
        {"name": "flash_d128_odd", "kind": "attention", "op": "flash", "heads": 32, "kv_heads": 32, "dim": 128,
         "seq": 1111, "prompts": 1},
        # A serving batch's attention over a long paged cache, lengths far apart.
        {"name": "paged_decode_64", "kind": "decode", "seqs": 64, "heads": 32, "kv_heads": 8, "dim": 128, "page": 16,
         "lo": 128, "hi": 4096},
        # Probabilities over a vocabulary.
        {"name": "softmax_vocab", "kind": "rows", "op": "softmax", "rows": 256, "cols": 32000},
        # A whole model: one decode step of a 32-sequence batch, logits out.
        {"name": "engine_decode_32", "kind": "engine", "mode": "decode", "model": "tinyllama", "layers": 22, "seqs": 32,
         "lo": 512, "hi": 639},
        # A prefill step of packed prompts of uneven lengths, logits of their last rows.
        {"name": "engine_prefill", "kind": "engine", "mode": "prefill", "model": "tinyllama", "layers": 8, "seqs": 4,
         "lo": 170, "hi": 255},
    ]


def _log(rng, lo, hi):
    """A whole number in lo .. hi, evenly over its logarithm."""
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _size(rng, lo, hi):
    """As `_log`; half of them as drawn (odd ones), the others multiples of 8 or 64."""
    n = _log(rng, lo, hi)
    step = rng.choice((1, 1, 8, 64))
    return max(lo, min(hi, (n + step - 1) // step * step))


def _drawn(rng):
    kind = rng.choice(("mlp", "head", "matmul", "attention", "decode", "rows", "engine"))
    if kind == "mlp":
        dim, ffn = rng.choice(BLOCKS)
        return {"kind": kind, "rows": _log(rng, 1, 1024), "dim": dim, "ffn": ffn}
    if kind == "head":
        rows = _log(rng, 1, 64)
        return {"kind": kind, "rows": rows, "tokens": rows + rng.randrange(0, 512), "dim": rng.choice((1024, 2048, 4096)),
                "vocab": rng.choice((4000, 32000))}
    if kind == "matmul":
        op = rng.choice(("matmul", "matmul", "matmul_f32", "linear"))
        hi = 2048 if op == "matmul_f32" else 4096
        return {"kind": kind, "op": op, "m": _size(rng, 16, hi), "n": _size(rng, 64, hi), "k": _size(rng, 64, hi)}
    if kind == "attention":
        op = rng.choice(("flash", "flash", "prefill"))
        heads, kv = (rng.choice((4, 16, 24, 32)), 0) if op == "flash" else rng.choice(((32, 4), (32, 8), (8, 2)))
        seq = _log(rng, 64, 4096 if op == "flash" else 2048)
        return {"kind": kind, "op": op, "heads": heads, "kv_heads": kv or heads, "dim": rng.choice((32, 64, 64, 128)),
                "seq": seq, "prompts": rng.randrange(1, 5) if op == "prefill" else 1}
    if kind == "decode":
        heads, kv = rng.choice(((32, 8), (32, 4), (32, 32), (16, 16), (8, 2), (16, 1)))
        hi = _log(rng, 64, 4096)
        return {"kind": kind, "seqs": _log(rng, 1, 64), "heads": heads, "kv_heads": kv, "dim": rng.choice((64, 128)),
                "page": rng.choice((16, 32)), "lo": max(1, hi // rng.choice((1, 4, 32))), "hi": hi}
    if kind == "rows":
        op = rng.choice(("softmax", "rmsnorm"))
        cols = _size(rng, 64, 32000 if op == "softmax" else 8192)
        return {"kind": kind, "op": op, "rows": _log(rng, 8, 8192), "cols": cols}
    mode = rng.choice(("decode", "prefill"))
    model = rng.choice(("tinyllama", "tinyllama", "tiny"))
    hi = _log(rng, 16, 240 if model == "tiny" else 639)
    return {"kind": kind, "mode": mode, "model": model, "layers": 2 if model == "tiny" else rng.randrange(2, 7),
            "seqs": _log(rng, 1, 32) if mode == "decode" else max(1, min(4, 1000 // hi)), "lo": max(1, hi // 2), "hi": hi}


def draw(rng):
    while True:
        case = _drawn(rng)
        w = work(case)
        if w["flops"] <= 1.37e11 and w["bytes"] <= 8e8:
            return case


# ---------------------------------------------------------------- inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, scale=1.0, dtype=torch.float16):
    return torch.randn(*shape, generator=g, device=DEV).mul_(scale).to(dtype)


def _uniform(g, *shape, scale=1.0, dtype=torch.float16):
    return torch.rand(*shape, generator=g, device=DEV).mul_(2.0).sub_(1.0).mul_(scale).to(dtype)


def _weight(g, rows, cols):
    """A projection as the engine's random weights have it: uniform, scaled by 1 / sqrt(columns)."""
    return _uniform(g, rows, cols, scale=cols ** -0.5)


def _pow2(n):
    return 1 << (int(n) - 1).bit_length()


class _State:
    """Launches in order, what they return, and (an engine's) what to close."""

    def __init__(self, calls=(), outputs=None, engine=None, step=None):
        self.calls, self.outputs, self.engine, self.step = list(calls), outputs, engine, step

    def __del__(self):
        if self.engine is not None:
            self.engine.close()


def _call(file, name, tensors, scalars=(), meta=()):
    k = T.kernel(file, name, [tuple(t.shape) for t in tensors], meta)
    return k, [T.Buf(t.data_ptr(), t.numel() * t.element_size()) for t in tensors] + list(scalars), tensors


def _empty(*shape, dtype=torch.float16):
    return torch.zeros(*shape, dtype=dtype, device=DEV)


# ---- one decoder MLP: the residual stream from the tokens' embeddings (so a
# pass can be repeated), its norm, gate_up and the down projection.

def _mlp_inputs(c, seed):
    g = _gen(seed)
    m, d, f = c["rows"], c["dim"], c["ffn"]
    tok = torch.randint(0, 4000, (m,), generator=g, device=DEV, dtype=torch.int32)
    return (tok, _uniform(g, 4000, d, scale=8 * d ** -0.5), _uniform(g, d, scale=0.2).add_(1.0), _weight(g, f, d),
            _weight(g, f, d), _weight(g, d, f))


def _mlp(c, seed):
    tok, emb, wn, wg, wu, wd = _mlp_inputs(c, seed)
    m, d, f = c["rows"], c["dim"], c["ffn"]
    x, h, y = _empty(m, d, dtype=torch.float32), _empty(m, d), _empty(m, f)
    calls = [_call("llm", "embed", [tok, emb, x]),
             _call("llm", "rmsnorm", [x, wn, h], [T.F32(1e-5)], [("BC", _pow2(d))]),
             _call("llm", "gate_up", [h, wg, wu, y]),
             _call("llm", "linear_residual", [y, wd, x])]
    return _State(calls, {"residual": x, "activations": y})


def _rms64(x, w, eps):
    return x / torch.sqrt(x.square().mean(-1, keepdim=True) + eps) * w.double()


def _mlp_exact(c, seed):
    tok, emb, wn, wg, wu, wd = _mlp_inputs(c, seed)
    x = emb[tok.long()].double()
    h = _rms64(x, wn, 1e-5)
    y = torch.nn.functional.silu(h @ wg.double().t()) * (h @ wu.double().t())
    return {"residual": x + y @ wd.double().t(), "activations": y}


def _mlp_work(c):
    m, d, f = c["rows"], c["dim"], c["ffn"]
    return {"bytes": 2.0 * 3 * d * f + m * (4.0 + 2 * d + 4 * d + 2 * f) + 2.0 * d, "flops": 6.0 * m * d * f}


# ---- the head: rmsnorm of the rows that want logits, and the output projection.

def _head_inputs(c, seed):
    g = _gen(seed)
    t, d = c["tokens"], c["dim"]
    idx = torch.randperm(t, generator=g, device=DEV)[: c["rows"]].to(torch.int32)
    return _normal(g, t, d, dtype=torch.float32), idx, _uniform(g, d, scale=0.2).add_(1.0), _weight(g, c["vocab"], d)


def _head(c, seed):
    x, idx, wn, w = _head_inputs(c, seed)
    h, y = _empty(c["rows"], c["dim"]), _empty(c["rows"], c["vocab"], dtype=torch.float32)
    calls = [_call("llm", "rmsnorm_rows", [x, idx, wn, h], [T.F32(1e-5)], [("BC", _pow2(c["dim"]))]),
             _call("llm", "logits", [h, w, y])]
    return _State(calls, {"logits": y})


def _head_exact(c, seed):
    x, idx, wn, w = _head_inputs(c, seed)
    return {"logits": _rms64(x[idx.long()].double(), wn, 1e-5) @ w.double().t()}


def _head_work(c):
    b, d, v = c["rows"], c["dim"], c["vocab"]
    return {"bytes": 2.0 * v * d + b * (4.0 * d + 4 + 4 * v) + 2.0 * d, "flops": 2.0 * b * d * v}


# ---- products: matmul (A B, f16), matmul_f32 (A B, f32), linear (X W^T + b).

def _matmul_inputs(c, seed):
    g = _gen(seed)
    m, n, k = c["m"], c["n"], c["k"]
    dt = torch.float32 if c["op"] == "matmul_f32" else torch.float16
    a = _normal(g, m, k, scale=k ** -0.5, dtype=dt)
    if c["op"] == "linear":
        return a, _normal(g, n, k), _uniform(g, n)
    return a, _normal(g, k, n, scale=1.0 if dt == torch.float32 else k ** -0.5, dtype=dt), None


def _matmul(c, seed):
    a, b, bias = _matmul_inputs(c, seed)
    y = _empty(c["m"], c["n"], dtype=a.dtype)
    return _State([_call("matmul", c["op"], [a, b, y] if bias is None else [a, b, bias, y])], y)


def _matmul_exact(c, seed):
    a, b, bias = _matmul_inputs(c, seed)
    if bias is not None:
        return a.double() @ b.double().t() + bias.double()
    return a.double() @ b.double()


def _matmul_work(c):
    m, n, k = c["m"], c["n"], c["k"]
    return {"bytes": (4.0 if c["op"] == "matmul_f32" else 2.0) * (m * k + k * n + m * n), "flops": 2.0 * m * n * k}


# ---- causal attention: flash_attention [H, S, D]; prefill_attention over
# packed prompts [S, H, D] with grouped kv heads.

def _lens(c, seed):
    """The prompts' lengths: seq rows cut at places of the seed's choice."""
    r = np.random.default_rng(seed)
    n = min(c["prompts"], c["seq"])
    cuts = np.sort(r.choice(np.arange(1, c["seq"]), n - 1, replace=False)) if n > 1 else np.zeros(0, np.int64)
    return np.diff(np.concatenate([[0], cuts, [c["seq"]]])).astype(int).tolist()


def _attention_inputs(c, seed):
    g = _gen(seed)
    h, kv, s, d = c["heads"], c["kv_heads"], c["seq"], c["dim"]
    if c["op"] == "flash":
        return tuple(_normal(g, h, s, d) for _ in range(3)) + (None,)
    starts, at = [], 0
    for n in _lens(c, seed):
        starts += [at] * n
        at += n
    return (_normal(g, s, h, d), _normal(g, s, kv, d), _normal(g, s, kv, d),
            torch.tensor(starts, dtype=torch.int32, device=DEV))


def _attention(c, seed):
    q, k, v, starts = _attention_inputs(c, seed)
    o, scale = torch.zeros_like(q), [T.F32(c["dim"] ** -0.5)]
    if starts is None:
        return _State([_call("attention", "flash_attention", [q, k, v, o], scale)], o)
    return _State([_call("llm", "prefill_attention", [q, k, v, starts, o], scale)], o)


def _causal64(q, k, v, scale):
    """Attention of one head's rows q [n, D] over the keys that end with them, in 64 bits."""
    n, m = q.shape[0], k.shape[0]
    s = (q.double() @ k.double().t()) * scale
    keep = torch.arange(m, device=DEV)[None, :] <= torch.arange(m - n, m, device=DEV)[:, None]
    return torch.softmax(s.masked_fill(~keep, -math.inf), -1) @ v.double()


def _attention_exact(c, seed):
    q, k, v, starts = _attention_inputs(c, seed)
    scale, rep = c["dim"] ** -0.5, c["heads"] // c["kv_heads"]
    if starts is None:
        return torch.stack([_causal64(q[h], k[h], v[h], scale) for h in range(c["heads"])])
    o, at = torch.zeros(q.shape, dtype=torch.float64, device=DEV), 0
    for n in _lens(c, seed):
        for h in range(c["heads"]):
            kh, vh = k[at:at + n, h // rep].contiguous(), v[at:at + n, h // rep].contiguous()
            o[at:at + n, h] = _causal64(q[at:at + n, h].contiguous(), kh, vh, scale)
        at += n
    return o


def _attention_work(c):
    h, kv, s, d = c["heads"], c["kv_heads"], c["seq"], c["dim"]
    # (the causal half of each prompt; packed prompts counted at even lengths)
    return {"bytes": 2.0 * s * d * (2 * h + 2 * kv), "flops": 2.0 * h * s * s * d / c["prompts"]}


# ---- decode attention over a paged cache: decode_attention (grouped kv
# heads) or paged_attention (a kv head per query head).

def _decode_inputs(c, seed):
    g, r = _gen(seed), np.random.default_rng(seed)
    b, h, kv, d, p = c["seqs"], c["heads"], c["kv_heads"], c["dim"], c["page"]
    lens = r.integers(c["lo"], c["hi"] + 1, b).astype(np.int32)
    need = (lens + p - 1) // p
    pages = int(need.sum())
    table = np.zeros((b, (c["hi"] + p - 1) // p), np.int32)
    perm, at = r.permutation(pages).astype(np.int32), 0
    for i, n in enumerate(need):
        table[i, :n] = perm[at:at + n]
        at += n
    return (_normal(g, b, h, d), _normal(g, pages, p, kv, d), _normal(g, pages, p, kv, d),
            torch.from_numpy(table).to(DEV), torch.from_numpy(lens).to(DEV))


def _decode(c, seed):
    q, kc, vc, table, lens = _decode_inputs(c, seed)
    o = torch.zeros_like(q)
    file, name = ("attention", "paged_attention") if c["heads"] == c["kv_heads"] else ("llm", "decode_attention")
    return _State([_call(file, name, [q, kc, vc, table, lens, o], [T.F32(c["dim"] ** -0.5)])], o)


def _decode_exact(c, seed):
    q, kc, vc, table, lens = _decode_inputs(c, seed)
    kv, d, rep = c["kv_heads"], c["dim"], c["heads"] // c["kv_heads"]
    o = torch.zeros(q.shape, dtype=torch.float64, device=DEV)
    for i, n in enumerate(lens.tolist()):
        rows = table[i, : (n + c["page"] - 1) // c["page"]].long()
        k, v = kc[rows].reshape(-1, kv, d)[:n].double(), vc[rows].reshape(-1, kv, d)[:n].double()
        for j in range(kv):
            hs = slice(j * rep, (j + 1) * rep)
            s = (q[i, hs].double() @ k[:, j].contiguous().t()) * d ** -0.5
            o[i, hs] = torch.softmax(s, -1) @ v[:, j].contiguous()
    return o


def _decode_work(c):
    tokens = c["seqs"] * (c["lo"] + c["hi"]) / 2.0
    b, h, kv, d = c["seqs"], c["heads"], c["kv_heads"], c["dim"]
    return {"bytes": tokens * kv * d * 4 + 4.0 * b * h * d + 4.0 * tokens / c["page"] + 4.0 * b,
            "flops": 4.0 * tokens * h * d}


# ---- row kernels: softmax (f32) and rmsnorm (f16).

def _rows_inputs(c, seed):
    g = _gen(seed)
    if c["op"] == "softmax":
        return _normal(g, c["rows"], c["cols"], scale=2.0, dtype=torch.float32), None
    return _normal(g, c["rows"], c["cols"]), _uniform(g, c["cols"], scale=0.2).add_(1.0)


def _rows(c, seed):
    x, w = _rows_inputs(c, seed)
    y = torch.zeros_like(x)
    meta = [("BR", 1), ("BC", _pow2(c["cols"]))]
    if w is None:
        return _State([_call("basic", "softmax", [x, y], (), meta)], y)
    return _State([_call("basic", "rmsnorm", [x, w, y], [T.F32(1e-5)], meta)], y)


def _rows_exact(c, seed):
    x, w = _rows_inputs(c, seed)
    return torch.softmax(x.double(), -1) if w is None else _rms64(x.double(), w, 1e-5)


def _rows_work(c):
    n = float(c["rows"]) * c["cols"]
    return {"bytes": (8.0 if c["op"] == "softmax" else 4.0) * n, "flops": 5.0 * n}


# ---- the engine: one step of a Llama-shaped decoder over its paged cache.

PAGE = 16


def _config(c):
    cfg = T.Config.tiny() if c["model"] == "tiny" else T.Config.tinyllama()
    cfg.layers = c["layers"]
    return cfg


def _layer_shapes(cfg):
    d, hd, f = cfg.dim, cfg.heads * cfg.head_dim, cfg.ffn
    return ((d,), (cfg.qkv(), d), (d, hd), (d,), (f, d), (f, d), (d, f))


def _model(cfg, seed):
    """Random weights, on the GPU: embedding, the layers' tensors, norm, head."""
    g = _gen(seed)
    layers = [[torch.ones(s, dtype=torch.float16, device=DEV) if len(s) == 1 else _weight(g, *s)
               for s in _layer_shapes(cfg)] for _ in range(cfg.layers)]
    embed = _uniform(g, cfg.vocab, cfg.dim, scale=8 * cfg.dim ** -0.5)
    return embed, layers, torch.ones(cfg.dim, dtype=torch.float16, device=DEV), _weight(g, cfg.vocab, cfg.dim)


def _prompts(c, cfg, seed):
    r = np.random.default_rng(seed)
    lens = r.integers(c["lo"], c["hi"] + 1, c["seqs"])
    return [r.integers(3, cfg.vocab, int(n)).tolist() for n in lens]


def _engine(c, seed):
    cfg, decode = _config(c), c["mode"] == "decode"
    embed, layers, norm, head = _model(cfg, seed)
    flat = torch.cat([t.reshape(-1) for layer in layers for t in layer])
    weights = [t.cpu().numpy().reshape(-1) for t in (embed, flat, norm, head)]
    del embed, layers, flat, norm, head
    prompts = _prompts(c, cfg, seed)
    per_seq = (c["hi"] + 1 + PAGE - 1) // PAGE
    tokens = max(c["hi"] if decode else sum(map(len, prompts)), c["seqs"])
    engine = T.Engine(cfg, T.Limits(PAGE, per_seq * c["seqs"], tokens, per_seq), weights)
    tables = np.random.default_rng(seed + 1).permutation(per_seq * c["seqs"]).reshape(c["seqs"], per_seq)

    def slot(i, p):
        return int(tables[i, p // PAGE]) * PAGE + p % PAGE

    if not decode:
        step = dict(tokens=sum(prompts, []), pos=[p for s in prompts for p in range(len(s))],
                    slots=[slot(i, p) for i, s in enumerate(prompts) for p in range(len(s))], mode=T.Engine.PACKED,
                    starts=np.repeat(np.cumsum([0] + [len(s) for s in prompts[:-1]]), [len(s) for s in prompts]),
                    want=(np.cumsum([len(s) for s in prompts]) - 1).tolist())
        return _State(engine=engine, step=_as_arrays(step))
    # Decode: every prompt but its last token is in the cache, one prefill step each.
    for i, s in enumerate(prompts):
        if len(s) > 1:
            n = len(s) - 1
            engine.step(s[:n], list(range(n)), [slot(i, p) for p in range(n)], T.Engine.PREFILL)
    step = dict(tokens=[s[-1] for s in prompts], pos=[len(s) - 1 for s in prompts],
                slots=[slot(i, len(s) - 1) for i, s in enumerate(prompts)], mode=T.Engine.DECODE, tables=tables,
                lens=[len(s) for s in prompts], want=range(c["seqs"]))
    return _State(engine=engine, step=_as_arrays(step))


def _as_arrays(step):
    return {k: v if k == "mode" else np.asarray(v, np.int32) for k, v in step.items()}


def _engine_exact(c, seed):
    cfg = _config(c)
    embed, layers, norm, head = _model(cfg, seed)
    prompts = _prompts(c, cfg, seed)
    lens = [len(s) for s in prompts]
    tok = torch.tensor(sum(prompts, []), device=DEV)
    pos = torch.cat([torch.arange(n, device=DEV) for n in lens]).double()
    h, kv, d = cfg.heads, cfg.kv_heads, cfg.head_dim
    inv = cfg.rope_theta ** (-torch.arange(0, d, 2, device=DEV).double() / d)
    cs, sn = torch.cos(pos[:, None] * inv)[:, None], torch.sin(pos[:, None] * inv)[:, None]

    def turned(t):
        a, b = t[..., : d // 2], t[..., d // 2:]
        return torch.cat([a * cs - b * sn, b * cs + a * sn], -1)

    x = embed[tok].double()
    for n1, wqkv, wo, n2, wg, wu, wd in layers:
        qkv = (_rms64(x, n1, cfg.eps) @ wqkv.double().t()).view(-1, h + 2 * kv, d)
        q, k, v = turned(qkv[:, :h]), turned(qkv[:, h:h + kv]), qkv[:, h + kv:]
        o, at = torch.empty_like(q), 0
        for n in lens:
            for i in range(h):
                j = i // (h // kv)
                o[at:at + n, i] = _causal64(q[at:at + n, i].contiguous(), k[at:at + n, j].contiguous(),
                                            v[at:at + n, j].contiguous(), d ** -0.5)
            at += n
        x = x + o.reshape(-1, h * d) @ wo.double().t()
        y = _rms64(x, n2, cfg.eps)
        x = x + (torch.nn.functional.silu(y @ wg.double().t()) * (y @ wu.double().t())) @ wd.double().t()
    last = torch.tensor(np.cumsum(lens) - 1, device=DEV)
    return _rms64(x[last], norm, cfg.eps) @ head.double().t()


def _engine_work(c):
    cfg, b = _config(c), c["seqs"]
    ctx = (c["lo"] + c["hi"]) / 2.0
    params = sum(math.prod(s) for s in _layer_shapes(cfg)) * cfg.layers
    kv_row = 4.0 * cfg.kv_heads * cfg.head_dim * cfg.layers  # K and V of one token, all layers
    rows, hd = (b, cfg.heads * cfg.head_dim) if c["mode"] == "decode" else (b * ctx, cfg.heads * cfg.head_dim)
    seen = b * ctx if c["mode"] == "decode" else b * ctx * ctx / 2  # (query, key) pairs
    return {"bytes": 2.0 * (params + cfg.vocab * cfg.dim) + b * ctx * kv_row + 4.0 * b * cfg.vocab + 2.0 * rows * cfg.dim,
            "flops": 2.0 * rows * params + 4.0 * seen * hd * cfg.layers + 2.0 * b * cfg.vocab * cfg.dim}


# ---------------------------------------------------------------- the interface

KINDS = {"mlp": (_mlp, _mlp_exact, _mlp_work), "head": (_head, _head_exact, _head_work),
         "matmul": (_matmul, _matmul_exact, _matmul_work), "attention": (_attention, _attention_exact, _attention_work),
         "decode": (_decode, _decode_exact, _decode_work), "rows": (_rows, _rows_exact, _rows_work),
         "engine": (_engine, _engine_exact, _engine_work)}


def prepare(case, seed):
    T.open()
    state = KINDS[case["kind"]][0](case, seed)
    torch.cuda.synchronize()  # the inputs come from torch's stream, the launches go to the library's
    return state


def run(state):
    if state.engine is not None:
        return state.engine.step(**state.step)
    for kernel, args, _ in state.calls:
        T.launch(kernel, args)
    return state.outputs


def exact(case, seed):
    return KINDS[case["kind"]][1](case, seed)


def work(case):
    return KINDS[case["kind"]][2](case)


def tolerance(case):
    """About four times the difference of the outputs from `exact` (rel), as
    measured over the listed cases and draws of each kind."""
    if case["kind"] == "rows" and case["op"] == "softmax":
        return {"rel": 1e-6, "max": 2e-5}  # (measured 1e-7)
    if case["kind"] == "matmul" and case["op"] == "matmul_f32":
        return {"rel": 4e-6, "max": 1e-4}  # (6e-7 at 1024 terms, growing with their root)
    if case["kind"] == "matmul":
        # Measured 2e-4 off `exact`; two passes of the 256 x 256 tiles over the
        # same inputs differed by 1.3e-3, 0.17 at most.
        return {"rel": 2e-3, "max": 0.5}
    if case["kind"] == "engine":
        return {"rel": 2.2e-3, "max": 0.05}  # (5.4e-4 over 22 layers)
    return {"rel": 1.5e-3, "max": 0.05}  # f16 outputs (2.1e-4 .. 3.6e-4)
