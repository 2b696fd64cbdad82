"""The calls whose speed counts, as a program on the device path makes them.

A serving process holds a context, its models and paged caches, and spends its
time in forward passes (prompt chunks, decode rows, verify rows), speculative
steps (greedy and sampled) and, at load time, in the quantizer and the AWQ
search. Each case is one such call, or the calls of one engine step, through
the public entry points of ferrolm_amd.gpu (and, for a product on device
buffers, fg_matmul_device of the C ABI).

`listed()` is a spread of them; `draw(rng)` gives others of the same ranges;
`prepare` makes what the program has in hand (models are kept per process, as
a server keeps them; contexts are prefilled with tokens made from the seed);
`run` is one pass and `exact` the same outputs in 64-bit torch without this
repository's kernels.

Weights are random with a trained model's scales: projections N(0, 0.02) (the
quantized ones as the codes and group scales such a matrix has), norm weights
log-uniform in [0.5, 2] (what the AWQ fold leaves), embeddings scaled so that
the logits have a standard deviation of about 3, which gives distributions
about as peaked as a language model's. Two such models seldom agree, so a
speculative step emits one token; its device work does not depend on that.
"""
from __future__ import annotations

import math
import zlib
from dataclasses import replace

import numpy as np
import torch

from ferrolm_amd import gpu
from ferrolm_amd.weights import BF16, INT4, INT8, HostModel, Layer, Matrix, shape

KINDS = {"bf16": BF16, "int8": INT8, "int4": INT4}
# The 8B shape runs 8 of its 32 layers (they are alike; all of them only take longer to make).
LAYERS = {"llama3-8b": 8}


def listed():
    return [
        # One decode row of a small bf16 model: a draft round, or a 135M model served alone. Launch-bound.
        dict(name="decode_135m_bf16", call="forward", model="smollm2-135m", weights="bf16", seqs=1, rows=1, lo=1000,
             hi=1000, logits="last"),
        # The verify rows of one stream on an int4 target, every row's logits on the host.
        dict(name="verify_1p7b_int4", call="forward", model="smollm2-1.7b", weights="int4", seqs=1, rows=4, lo=1030,
             hi=1030, logits="all"),
        # A whole prompt (time to first token) through the target, and one of odd length through the draft.
        dict(name="prefill_1p7b_int4", call="forward", model="smollm2-1.7b", weights="int4", seqs=1, rows=1024, lo=0,
             hi=0, logits="last"),
        dict(name="prefill_135m_bf16", call="forward", model="smollm2-135m", weights="bf16", seqs=1, rows=777, lo=0,
             hi=0, logits="last"),
        # Verify rows of 16 streams on a grouped-query model at head dim 128, then one stream's plain step.
        dict(name="verify_8b_int4_b16", call="verify", model="llama3-8b", weights="int4", seqs=16, rows=5, lo=512,
             hi=4001),
        # The latency-bound headline: one greedy stream, three proposals, then its next plain step.
        dict(name="spec_1p7b_int4_b1", call="spec", model="smollm2-1.7b", weights="int4", draft="smollm2-135m", k=3,
             seqs=1, lo=1030, hi=1030, temperature=0.0, top_p=1.0, top_k=0),
        # A full batch of greedy streams with ragged contexts over shuffled cache blocks.
        dict(name="spec_1p7b_int8_b32", call="spec", model="smollm2-1.7b", weights="int8", draft="smollm2-135m", k=4,
             seqs=32, lo=128, hi=2048, temperature=0.0, top_p=1.0, top_k=0),
        # Sampled streams at the usual chat settings, no top-k limit, beside one request's plain step.
        dict(name="spec_sampled_360m_int8_b4", call="spec", model="smollm2-360m", weights="int8",
             draft="smollm2-135m", k=4, seqs=4, lo=200, hi=700, temperature=0.8, top_p=0.95, top_k=0),
        # One projection alone on device buffers: a decode step's down, a batched verify's gate/up.
        dict(name="matmul_int4_m4", call="matmul", weights="int4", n=2048, k=8192, m=4),
        dict(name="matmul_int8_m160", call="matmul", weights="int8", n=16384, k=2048, m=160),
        # Load time: quantizing one matrix, and the AWQ search of one projection.
        dict(name="quantize_int4", call="quantize", weights="int4", n=16384, k=2048),
        dict(name="awq_search_int4", call="awq", weights="int4", n=6144, k=2048, m=256),
    ]


def draw(rng):
    def size(lo, hi):
        """Log-uniform in [lo, hi]."""
        return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))

    what = rng.choice(("decode", "decode", "prefill", "prefill", "verify", "spec", "spec", "sampled", "matmul",
                       "matmul", "quantize", "awq"))
    model, weights = rng.choice((("smollm2-135m", "bf16"), ("smollm2-360m", "int8"), ("smollm2-1.7b", "int4"),
                                 ("smollm2-1.7b", "int8")))
    lo = size(16, 1500)
    ctx = dict(lo=lo, hi=rng.randint(lo, 2000))
    if what == "decode":
        return dict(call="forward", model=model, weights=weights, seqs=size(1, 24), rows=1, logits="last", **ctx)
    if what == "prefill":
        return dict(call="forward", model=model, weights=weights, seqs=1, rows=size(20, 1024),
                    lo=rng.choice((0, 0, size(16, 900))), hi=0, logits="last")
    if what == "verify":
        if rng.random() < 0.3:
            model, weights = "llama3-8b", "int4"
        return dict(call="verify", model=model, weights=weights, seqs=size(1, 16), rows=rng.randint(2, 6), **ctx)
    if what in ("spec", "sampled"):
        case = dict(call="spec", model=model, weights=weights, draft="smollm2-135m", k=rng.randint(1, 5), **ctx)
        if what == "spec":
            return dict(case, seqs=size(1, 24), temperature=0.0, top_p=1.0, top_k=0)
        return dict(case, k=rng.randint(1, 4), seqs=size(1, 4), temperature=rng.choice((0.6, 0.8, 1.0)),
                    top_p=rng.choice((0.9, 0.95, 1.0)), top_k=rng.choice((0, 0, 20, 50, 2000)))
    weights = rng.choice(("int4", "int8") if what in ("quantize", "awq") else ("int4", "int8", "bf16"))
    if what == "matmul":
        n, k = rng.choice(((2048, 2048), (6144, 2048), (16384, 2048), (2048, 8192), (960, 2560), (1536, 576),
                           (4096, 4096), (6144, 4096)))
        return dict(call="matmul", weights=weights, n=n, k=k, m=size(1, 1024))
    n, k = 32 * size(8, 192), 32 * size(8, 64)
    if what == "quantize":
        return dict(call="quantize", weights=weights, n=n, k=k)
    return dict(call="awq", weights=weights, n=n, k=k, m=size(16, 256))


# ---------------------------------------------------------------------------
# Models
# ---------------------------------------------------------------------------
_ctx = None
_models = {}


def _context():
    global _ctx
    if _ctx is None:
        _ctx = gpu.Context(0)
    return _ctx


def _config(name):
    c = shape(name)
    return replace(c, layers=LAYERS.get(name, c.layers))


def _rand(*key):
    """A device generator of its own for each key."""
    g = torch.Generator("cuda")
    g.manual_seed(zlib.crc32(repr(key).encode()))
    return g


def _codes(kind, n, k, *key):
    """The codes [n][k] and group scales [n][k / 32] of a quantized N(0, 0.02) matrix."""
    g = _rand(kind, n, k, *key)
    half, spread = (8, 3.5) if kind == INT4 else (128, 42.0)
    q = torch.randn(n, k, generator=g, device="cuda").mul_(spread).round_().clamp_(1 - half, half - 1).to(torch.int8)
    s = (0.7 + 0.6 * torch.rand(n, k // 32, generator=g, device="cuda")) * (0.02 / spread)
    return q, s


def _bf16(n, k, std, *key):
    return (torch.randn(n, k, generator=_rand(n, k, *key), device="cuda") * std).to(torch.bfloat16)


def _dense64(kind, n, k, *key):
    if kind == BF16:
        return _bf16(n, k, 0.02, *key).double()
    q, s = _codes(kind, n, k, *key)
    return q.double() * s.double().repeat_interleave(32, dim=1)


def _matrix(kind, n, k, *key):
    """The same matrix as the library takes it."""
    if kind == BF16:
        return Matrix(BF16, n, k, bf16=_bf16(n, k, 0.02, *key).view(torch.uint16).cpu().numpy())
    q, s = _codes(kind, n, k, *key)
    p = q.view(n // 32, 32, k).transpose(1, 2)
    if kind == INT4:
        u = (p + 8).to(torch.uint8)
        p = u[..., :16] | (u[..., 16:] << 4)
    sc = s.view(n // 32, 32, k // 32).transpose(1, 2).contiguous()
    return Matrix(kind, n, k, q=p.contiguous().view(torch.uint8).flatten().cpu().numpy(),
                  s=sc.flatten().cpu().numpy())


def _norm(h, *key):
    return torch.exp((2 * torch.rand(h, generator=_rand(h, *key), device="cuda") - 1) * math.log(2.0))


def _projections(c):
    return (("wqkv", c.qkv_dim, c.hidden), ("wo", c.hidden, c.q_dim), ("w_gate_up", 2 * c.intermediate, c.hidden),
            ("w_down", c.hidden, c.intermediate))


def _embedding(name, which):
    c = _config(name)
    return _bf16(c.vocab, c.hidden, 3.0 / math.sqrt(c.hidden), name, which)


def _model(name, weights):
    if (name, weights) not in _models:
        c, kind = _config(name), KINDS[weights]
        layers = []
        for l in range(c.layers):
            mats = {w: _matrix(kind, n, k, name, l, w) for w, n, k in _projections(c)}
            layers.append(Layer(attn_norm=_norm(c.hidden, name, l, 0).cpu().numpy(), bqkv=None,
                                mlp_norm=_norm(c.hidden, name, l, 1).cpu().numpy(), **mats))
        host = HostModel(cfg=c, embed=_embedding(name, "embed").view(torch.uint16).cpu().numpy(),
                         norm=np.ones(c.hidden, np.float32), layers=layers,
                         lm_head=None if c.tie_embeddings else
                         _embedding(name, "head").view(torch.uint16).cpu().numpy())
        _models[name, weights] = gpu.Model(_context(), host)
    return _models[name, weights]


# ---------------------------------------------------------------------------
# Sequences
# ---------------------------------------------------------------------------
def _lengths(case):
    """The context lengths of the case's sequences: spread evenly over [lo, hi], most of them odd or ragged."""
    n, lo, hi = case["seqs"], case["lo"], max(case["lo"], case["hi"])
    return [lo + (hi - lo) * i // max(1, n - 1) for i in range(n)]


def _tokens(case, seed, i, n):
    """n token ids of the case's i-th sequence."""
    return np.random.default_rng((seed, i)).integers(0, _config(case["model"]).vocab, n).astype(np.uint32)


def _sequences(case):
    """(context length, new tokens that the program gives) of each sequence, a plain step's own one last."""
    new = 1 if case["call"] == "spec" else case["rows"]
    seqs = [(n, new) for n in _lengths(case)]
    if case["call"] == "spec" and case["temperature"] > 0:
        seqs.append((case["lo"], 1))
    return seqs


def _tables(lengths, seed):
    """Block tables out of a shuffled pool, as a server's pool is after some requests, and the pool's size."""
    need = [(n + 15) // 16 for n in lengths]
    order = np.random.default_rng((seed, 7)).permutation(sum(need)).astype(np.uint32)
    ends = np.cumsum(need)
    return [order[e - n:e] for e, n in zip(ends, need)], sum(need)


def _prefilled(model, tokens, lengths, room, seed):
    """A cache holding the first lengths[i] of each sequence's tokens, and the block tables."""
    tables, blocks = _tables([n + room for n in lengths], seed)
    kv = gpu.KvCache(_context(), model.cfg, blocks)
    torch.cuda.synchronize()  # the new cache is cleared on a stream of its own
    chunks, rows = [], 0
    for t, n, b in zip(tokens, lengths, tables):
        for p in range(0, n, 2048):
            m = min(2048, n - p)
            if chunks and rows + m > 2048:
                gpu.forward(_context(), model, kv, chunks, logits=False)
                chunks, rows = [], 0
            chunks.append((t[p:p + m], p, b, gpu.LOGITS_NONE))
            rows += m
    if chunks:
        gpu.forward(_context(), model, kv, chunks, logits=False)
    return kv, tables


# ---------------------------------------------------------------------------
# The cases
# ---------------------------------------------------------------------------
def prepare(case, seed):
    call = case["call"]
    if call == "matmul":
        n, k, m = case["n"], case["k"], case["m"]
        kind = KINDS[case["weights"]]
        if (kind, n, k) not in _models:
            _models[kind, n, k] = gpu.Mat(_context(), _matrix(kind, n, k, "lone"))
        x = _activations(case, seed)
        state = dict(call=call, mat=_models[kind, n, k], x=x, m=m, y=torch.empty(m, n, device="cuda"))
        torch.cuda.synchronize()
        return state
    if call in ("quantize", "awq"):
        g = _rand(seed, "load")
        n, k = case["n"], case["k"]
        state = dict(call=call, kind=KINDS[case["weights"]],
                     w=(torch.randn(n, k, generator=g, device="cuda") * 0.02).cpu().numpy())
        if call == "awq":
            state["cal"] = _activations(case, seed).cpu().numpy()
        else:
            state["importance"] = torch.rand(k, generator=g, device="cuda").add_(0.1).square_().cpu().numpy()
        return state

    model = _model(case["model"], case["weights"])
    seqs = _sequences(case)
    lengths = [n for n, _ in seqs]
    tokens = [_tokens(case, seed, i, n + new) for i, (n, new) in enumerate(seqs)]
    room = 16 + case.get("rows", 0)
    kv, tables = _prefilled(model, tokens, lengths, room, seed)
    state = dict(call=call, model=model, kv=kv)
    if call == "spec":
        draft = _model(case["draft"], "bf16")
        dkv, dtables = _prefilled(draft, tokens, lengths, 16, seed + 1)
        state.update(draft=draft, dkv=dkv, k=case["k"], tables=tables, pos=lengths, plain=None, params=None, rng=None)
        b = case["seqs"]
        state["seqs"] = [gpu.SpecSeq(tail=t[-1:], draft_pos=n, pos=n, blocks=tb, draft_blocks=db)
                         for t, n, tb, db in zip(tokens[:b], lengths, tables, dtables)]
        if case["temperature"] > 0:
            state["params"] = [gpu.SamplingParams(case["temperature"], case["top_p"], case["top_k"])] * b
            state["rng"] = np.array([gpu.rng_init(seed + 1 + i) for i in range(b)], np.uint64)
            state["plain"] = (tokens[b][-1:], lengths[b], tables[b], gpu.LOGITS_LAST)
        return state
    mode = gpu.LOGITS_LAST if call == "forward" and case["logits"] == "last" else gpu.LOGITS_ALL
    state["chunks"] = [(t[n:], n, b, mode) for t, n, b in zip(tokens, lengths, tables)]
    return state


def _activations(case, seed):
    """Rows of a projection's input: N(0, 1) with 1% of the channels 20 times as large."""
    x = torch.randn(case["m"], case["k"], generator=_rand(seed, "x"), device="cuda")
    x[:, torch.randperm(case["k"], generator=_rand(seed, "channels"), device="cuda")[:max(1, case["k"] // 100)]] *= 20
    return x


def run(state):
    ctx, call = _context(), state["call"]
    if call == "forward":
        o = gpu.forward(ctx, state["model"], state["kv"], state["chunks"])
        return {"logits": o.logits, "argmax": o.argmax.astype(np.int64)}
    if call == "verify":
        # the verify pass, then the plain step of the first sequence from the token its last row gave
        o = gpu.forward(ctx, state["model"], state["kv"], state["chunks"], logits=False)
        tok, pos, blocks, _ = state["chunks"][0]
        p = gpu.forward(ctx, state["model"], state["kv"],
                        [(o.argmax[len(tok) - 1:len(tok)], pos + len(tok), blocks, gpu.LOGITS_LAST)])
        return {"argmax": o.argmax.astype(np.int64), "logits": p.logits}
    if call == "spec":
        rng = None if state["rng"] is None else state["rng"].copy()
        toks, acc = gpu.spec_step(ctx, state["model"], state["kv"], state["draft"], state["dkv"], state["seqs"],
                                  state["k"], state["params"], rng)
        # sampled: another request's plain step, as the engine runs it beside the sampled ones;
        # greedy: the first stream's own next step, too near its end to speculate again
        plain = state["plain"] or (toks[0][-1:], state["pos"][0] + len(toks[0]), state["tables"][0], gpu.LOGITS_LAST)
        p = gpu.forward(ctx, state["model"], state["kv"], [plain])
        out = {"tokens": np.concatenate(toks).astype(np.int64), "accepted": acc, "logits": p.logits}
        if rng is not None:
            out["rng"] = rng.view(np.int64)
        return out
    if call == "matmul":
        gpu.check(gpu.lib().fg_matmul_device(ctx.h, state["mat"].h, state["x"].data_ptr(), state["m"],
                                             state["y"].data_ptr()))
        return state["y"]
    if call == "quantize":
        m = gpu.quantize(ctx, state["kind"], state["w"], state["importance"])
        return {"codes": m.q, "scales": m.s}
    sc, alpha, plain, awq, m = gpu.awq_search(ctx, state["kind"], state["w"], state["cal"])
    return {"scales": sc, "alpha": alpha, "error_plain": plain, "error_awq": awq, "codes": m.q, "group_scales": m.s}


def _weight_bytes(kind, n, k):
    return n * k * {BF16: 2.0, INT8: 1.125, INT4: 0.625}[kind]


def _pass_work(c, kind, chunks, logit_rows):
    """Bytes and flops of one forward over chunks of (context, rows): every weight once, each sequence's keys
    and values once, the new ones written, the logits rows' head."""
    rows = sum(r for _, r in chunks)
    by = sum(_weight_bytes(kind, n, k) for _, n, k in _projections(c)) * c.layers
    fl = sum(2.0 * rows * n * k for _, n, k in _projections(c)) * c.layers
    kv = 2 * c.kv_heads * c.head_dim * 4
    by += c.layers * kv * sum(n + 2 * r for n, r in chunks)
    fl += c.layers * 4.0 * c.heads * c.head_dim * sum(r * n + r * (r + 1) / 2 for n, r in chunks)
    if logit_rows:
        by += 2.0 * c.vocab * c.hidden
        fl += 2.0 * logit_rows * c.vocab * c.hidden
    return np.array([by, fl])


def work(case):
    call = case["call"]
    if call == "matmul":
        n, k, m = case["n"], case["k"], case["m"]
        return dict(bytes=_weight_bytes(KINDS[case["weights"]], n, k) + 4.0 * m * (n + k), flops=2.0 * m * n * k)
    if call in ("quantize", "awq"):
        n, k = case["n"], case["k"]
        by = 4.0 * n * k + _weight_bytes(KINDS[case["weights"]], n, k)
        if call == "quantize":
            return dict(bytes=by, flops=4.0 * n * k * (11 if case["weights"] == "int4" else 6))
        return dict(bytes=by + 4.0 * case["m"] * k, flops=2.0 * case["m"] * n * k * 12)
    c, kind = _config(case["model"]), KINDS[case["weights"]]
    lengths = _lengths(case)
    if call == "forward":
        chunks = [(n, case["rows"]) for n in lengths]
        rows = len(chunks) if case["logits"] == "last" else sum(r for _, r in chunks)
        w = _pass_work(c, kind, chunks, rows) + [4.0 * rows * c.vocab, 0]
    elif call == "verify":
        chunks = [(n, case["rows"]) for n in lengths]
        w = _pass_work(c, kind, chunks, sum(r for _, r in chunks))
        w = w + _pass_work(c, kind, [(lengths[0] + case["rows"], 1)], 1) + [4.0 * c.vocab, 0]
    else:
        d, k = _config(case["draft"]), case["k"]
        w = _pass_work(c, kind, [(n, k + 1) for n in lengths], len(lengths) * (k + 1))
        for r in range(k):
            w = w + _pass_work(d, BF16, [(n + r, 1) for n in lengths], len(lengths))
        w = w + _pass_work(c, kind, [(case["lo"], 1)], 1) + [4.0 * c.vocab, 0]
    return dict(bytes=float(w[0]), flops=float(w[1]))


def tolerance(case):
    # Whole numbers (tokens, counts, codes, generator states) are the same everywhere. The quantizer and the
    # search are specified bit for bit.
    if case["call"] in ("quantize", "awq"):
        return "exact"
    # A lone product: f32 sums of products of inputs held to 16 bits or more (16 rows and up; measured against 64
    # bits: 2.5e-6) or to 29 bits (fewer rows; 1.1e-7).
    if case["call"] == "matmul":
        return {"rel": 1e-5, "max": 1e-4}
    # A whole model: 32-bit sums and 16-bit pairs of activations through every layer (measured against 64 bits:
    # 4e-6 to 3e-5).
    return {"rel": 1e-4, "max": 1e-3}


# ---------------------------------------------------------------------------
# The same in 64 bits
# ---------------------------------------------------------------------------
def _rope(c, n):
    """cos and sin of the angles, which are f32 by specification."""
    f = (1.0 / np.float32(float(c.rope_theta) ** (np.arange(0, c.head_dim, 2) / c.head_dim))).astype(np.float32)
    a = torch.from_numpy(np.arange(n, dtype=np.float32)[:, None] * f[None, :]).cuda().double()
    return torch.cos(a)[:, None, :], torch.sin(a)[:, None, :]


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat((a * cos - b * sin, b * cos + a * sin), dim=-1)


def _logits64(name, weights, tokens, rows):
    """Logits of the last `rows` of one sequence's tokens."""
    c, kind, n = _config(name), KINDS[weights], len(tokens)
    t = torch.from_numpy(np.asarray(tokens, np.int64)).cuda()
    embed = _embedding(name, "embed")
    x = embed[t].double()
    cos, sin = _rope(c, n)
    group = c.heads // c.kv_heads

    def normed(v):
        return v / torch.sqrt(v.square().mean(dim=1, keepdim=True) + c.rms_eps)

    for l in range(c.layers):
        w = {k: _dense64(kind, a, b, name, l, k) for k, a, b in _projections(c)}
        qkv = (normed(x) * _norm(c.hidden, name, l, 0).double()) @ w["wqkv"].T
        q, k, v = (a.reshape(n, -1, c.head_dim) for a in
                   qkv.split((c.q_dim, c.kv_heads * c.head_dim, c.kv_heads * c.head_dim), dim=1))
        q, k = _rotate(q, cos, sin), _rotate(k, cos, sin)
        out = torch.empty_like(q)
        hidden = torch.ones(n, n, dtype=torch.bool, device="cuda").triu_(1)
        for h in range(c.heads):
            s = (q[:, h] @ k[:, h // group].T / math.sqrt(c.head_dim)).masked_fill_(hidden, -math.inf)
            out[:, h] = torch.softmax(s, dim=1) @ v[:, h // group]
        x = x + out.reshape(n, -1) @ w["wo"].T
        gate, up = ((normed(x) * _norm(c.hidden, name, l, 1).double()) @ w["w_gate_up"].T).chunk(2, dim=1)
        x = x + (gate / (1 + torch.exp(-gate)) * up) @ w["w_down"].T
    head = embed if c.tie_embeddings else _embedding(name, "head")
    return (normed(x[n - rows:]) @ head.double().T).cpu().numpy()


def _greedy_step64(case, tokens):
    """The tokens that a greedy speculative step emits for one sequence."""
    ids = [int(t) for t in tokens]
    for _ in range(case["k"]):
        ids.append(int(_logits64(case["draft"], "bf16", ids, 1)[0].argmax()))
    best = _logits64(case["model"], case["weights"], ids, case["k"] + 1).argmax(axis=1)
    out = []
    for j in range(case["k"] + 1):
        out.append(int(best[j]))
        if j == case["k"] or out[-1] != ids[len(tokens) + j]:
            return out


def exact(case, seed):
    call = case["call"]
    if call in ("quantize", "awq"):
        return None  # defined bit for bit in 32-bit steps, and compared exactly
    if call == "matmul":
        w = _dense64(KINDS[case["weights"]], case["n"], case["k"], "lone")
        return _activations(case, seed).double() @ w.T
    name, weights = case["model"], case["weights"]
    seqs = _sequences(case)
    tokens = [_tokens(case, seed, i, n + new) for i, (n, new) in enumerate(seqs)]
    if call == "forward":
        if sum(len(t) for t in tokens) > 20000:
            return None
        rows = 1 if case["logits"] == "last" else case["rows"]
        return {"argmax": None, "logits": np.concatenate([_logits64(name, weights, t, rows) for t in tokens])}
    if call == "verify":
        nxt = _logits64(name, weights, tokens[0], 1)[0].argmax()
        return {"argmax": None, "logits": _logits64(name, weights, list(tokens[0]) + [nxt], 1)}
    if case["temperature"] > 0:
        return {"tokens": None, "accepted": None, "rng": None, "logits": _logits64(name, weights, tokens[-1], 1)}
    emitted = _greedy_step64(case, tokens[0])
    return {"tokens": None, "accepted": None, "logits": _logits64(name, weights, list(tokens[0]) + emitted, 1)}
