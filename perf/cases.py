"""Performance cases of the tecoops operator path: what an LLM serving program
has it do, through the public entry points, from the calls of one decode step
over a few sequences to a full prefill.

listed() holds the cases, draw() more of the same ranges.  prepare() makes
what a program has in hand before the call (weights, paged caches, block
tables, positions, output buffers), run() is one pass, exact() the same pass
in 64-bit torch, work() the bytes and operations the pass cannot do without.
Sizes come from the repository's benchmark and tests: hidden 4096, 32 query
and 8 kv heads of 128, weights [14336, 4096] and [4096, 14336], 64 decoding
sequences of 512..8192 keys, a 4 x 4096 prefill, 8192-token prefill batches.

Kinds of case:
  tokens   the small ops around attention over a batch of tokens: rms_norm
           with the fused residual add, then rotary on q and k with k and v
           stored into the paged cache (tokens = 1 per decoding sequence, or
           a prefill batch)
  conv     causal_conv1d over ragged sequences with conv state
  linear   the weight products of one decoder layer for `batch` tokens: qkv,
           attention output, gate + up, down
  attn     paged attention: q_lo..q_hi new tokens per sequence over
           ctx_lo..ctx_hi tokens already cached (q = 1: decode)
  block    the attention half of a decoder layer at a decode step, captured
           in a HIP graph and replayed: norm, q and kv products, rotary and
           cache store, attention, output product, residual norm
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))),
                                "teco-ops_amd"))
import tecoops  # noqa: E402

DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16}
EPS = 1e-6


def listed():
    return [
        # One decode step's small ops for 4 sequences, called one by one from
        # Python: the smallest calls, launch and host latency.
        dict(name="decode_tokens", kind="tokens", tokens=4, hidden=4096, heads=32, kv_heads=8,
             head=128, block=16, neox=True, dtype="f16", lens=1),
        # A prefill batch's 8192 tokens through the same ops: streaming.
        dict(name="prefill_tokens", kind="tokens", tokens=8192, hidden=4096, heads=32, kv_heads=8,
             head=128, block=16, neox=True, dtype="bf16", lens=2),
        # The convolution of a prefill batch of ragged prompts, in the
        # [dim, tokens] layout of the torch entry point; half the sequences
        # continue from a saved state.
        dict(name="conv_ragged", kind="conv", batch=16, dim=4096, width=4, len_lo=64, len_hi=2048,
             layout="rows", lens=3),
        # The weight products of a layer when one sequence decodes.
        dict(name="linear_f16_b1", kind="linear", batch=1, hidden=4096, heads=32, kv_heads=8,
             head=128, inter=14336, dtype="f16"),
        # The same with int8 weights for 8 sequences.
        dict(name="linear_i8_b8", kind="linear", batch=8, hidden=4096, heads=32, kv_heads=8,
             head=128, inter=14336, dtype="i8"),
        # A busy server's decode batch.
        dict(name="linear_bf16_b32", kind="linear", batch=32, hidden=4096, heads=32, kv_heads=8,
             head=128, inter=14336, dtype="bf16"),
        # Decode attention for a few sequences of moderate length.
        dict(name="attn_decode_b4", kind="attn", batch=4, q_lo=1, q_hi=1, ctx_lo=255, ctx_hi=4095,
             heads=32, kv_heads=8, head=128, block=16, dtype="f16", lens=4),
        # Decode attention for a full batch of long sequences.
        dict(name="attn_decode_b64", kind="attn", batch=64, q_lo=1, q_hi=1, ctx_lo=511,
             ctx_hi=8191, heads=32, kv_heads=8, head=128, block=16, dtype="bf16", lens=5),
        # Chunked prefill and multi-turn prompts: short query ranges over a
        # long cached context.
        dict(name="attn_chunks", kind="attn", batch=16, q_lo=16, q_hi=256, ctx_lo=512, ctx_hi=7936,
             heads=32, kv_heads=8, head=128, block=16, dtype="bf16", lens=6),
        # A batch of fresh prompts of mixed length.
        dict(name="attn_prompts", kind="attn", batch=24, q_lo=16, q_hi=1024, ctx_lo=0, ctx_hi=0,
             heads=32, kv_heads=8, head=128, block=16, dtype="f16", lens=7),
        # The long prefill: 4 prompts of 4096 tokens.
        dict(name="attn_prefill_4x4096", kind="attn", batch=4, q_lo=4096, q_hi=4096, ctx_lo=0,
             ctx_hi=0, heads=32, kv_heads=8, head=128, block=16, dtype="bf16", lens=8),
        # A whole decode step of a layer's attention half, as a server replays
        # it from a captured graph.
        dict(name="decode_block_b8", kind="block", batch=8, hidden=4096, heads=32, kv_heads=8,
             head=128, block=16, ctx_lo=255, ctx_hi=2047, dtype="f16", lens=9),
    ]


# ----------------------------------------------------------------- drawing

HEADS = [(32, 8), (32, 8), (16, 2), (16, 4), (16, 8), (40, 8), (64, 8), (32, 32)]
MOST_BYTES, MOST_FLOPS = 1.1e9, 5.5e11  # the largest listed cases


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw_once(rng):
    kind = rng.choice(["tokens", "conv", "linear", "linear", "attn", "attn", "attn", "block"])
    heads, kv_heads = rng.choice(HEADS)
    head = rng.choice([64, 96, 128, 128, 128])
    dtype = rng.choice(["f16", "bf16"])
    block = rng.choice([16, 16, 32, 64])
    lens = rng.randrange(1 << 20)
    hidden = 64 * rng.randint(16, 128)
    if kind == "tokens":
        return dict(kind=kind, tokens=_log(rng, 1, 8192), hidden=hidden, heads=heads,
                    kv_heads=kv_heads, head=head, block=block, neox=rng.random() < 0.75,
                    dtype=dtype, lens=lens)
    if kind == "conv":
        lo = _log(rng, 1, 512)
        return dict(kind=kind, batch=_log(rng, 1, 64), dim=8 * rng.randint(128, 1024),
                    width=rng.choice([4, 4, 3, 2]), len_lo=lo, len_hi=_log(rng, lo, 4096),
                    layout=rng.choice(["rows", "rows", "tokens"]), lens=lens)
    if kind == "linear":
        return dict(kind=kind, batch=_log(rng, 1, 64), hidden=hidden, heads=heads,
                    kv_heads=kv_heads, head=head, inter=64 * rng.randint(32, 256),
                    dtype=rng.choice(["f16", "bf16", "i8"]))
    if kind == "attn":
        how = rng.choice(["decode", "decode", "chunks", "prompts"])
        if how == "decode":
            q_lo = q_hi = 1
            ctx_lo = _log(rng, 16, 4096)
            ctx_hi = _log(rng, ctx_lo, 32768)
        elif how == "chunks":
            q_lo = _log(rng, 2, 256)
            q_hi = _log(rng, q_lo, 512)
            ctx_lo = _log(rng, 64, 4096)
            ctx_hi = _log(rng, ctx_lo, 8192)
        else:
            q_lo = _log(rng, 8, 2048)
            q_hi = _log(rng, q_lo, 8192)
            ctx_lo = ctx_hi = 0
        return dict(kind=kind, batch=_log(rng, 1, 64), q_lo=q_lo, q_hi=q_hi, ctx_lo=ctx_lo,
                    ctx_hi=ctx_hi, heads=heads, kv_heads=kv_heads, head=head, block=block,
                    dtype=dtype, lens=lens)
    ctx_lo = _log(rng, 16, 1024)
    return dict(kind=kind, batch=_log(rng, 1, 32), hidden=hidden, heads=heads, kv_heads=kv_heads,
                head=head, block=block, ctx_lo=ctx_lo, ctx_hi=_log(rng, ctx_lo, 4096),
                dtype=dtype, lens=lens)


def draw(rng):
    while True:
        c = _draw_once(rng)
        w = work(c)
        if w["bytes"] <= MOST_BYTES and w["flops"] <= MOST_FLOPS:
            return c


# ------------------------------------------------------------ sizes of a case

def _lengths(c):
    """(new tokens, cached tokens) of each sequence."""
    r = random.Random(c["lens"])

    def pick(lo, hi):
        return lo if lo == hi else _log(r, max(lo, 1), hi)

    if c["kind"] == "conv":
        return [pick(c["len_lo"], c["len_hi"]) for _ in range(c["batch"])], None
    if c["kind"] == "block":
        return [1] * c["batch"], [pick(c["ctx_lo"], c["ctx_hi"]) for _ in range(c["batch"])]
    # decode contexts spread evenly, other lengths over their logarithm
    q = [pick(c["q_lo"], c["q_hi"]) for _ in range(c["batch"])]
    if c["q_hi"] == 1:
        ctx = [r.randint(c["ctx_lo"], c["ctx_hi"]) for _ in range(c["batch"])]
    else:
        ctx = [pick(c["ctx_lo"], c["ctx_hi"]) for _ in range(c["batch"])]
    return q, ctx


def _linear_shapes(c):
    """(name, N, K) of a layer's weights."""
    attn = c["heads"] * c["head"]
    return [("qkv", attn + 2 * c["kv_heads"] * c["head"], c["hidden"]), ("o", c["hidden"], attn),
            ("gate_up", 2 * c["inter"], c["hidden"]), ("down", c["hidden"], c["inter"])]


def work(c):
    """Bytes and operations of one pass that it cannot do without."""
    if c["kind"] == "tokens":
        t, hid = c["tokens"], c["hidden"]
        kv = c["kv_heads"] * c["head"]
        rows = t * (4 * hid + 2 * c["heads"] * c["head"] + 4 * kv) + hid
        return {"bytes": 2 * rows + t * (16 + 4 * c["head"]), "flops": 0}
    if c["kind"] == "conv":
        n, _ = _lengths(c)
        state = c["batch"] * (c["width"] - 1) * c["dim"]
        return {"bytes": 2 * (2 * sum(n) * c["dim"] + 2 * state + c["width"] * c["dim"]),
                "flops": 2 * sum(n) * c["dim"] * c["width"]}
    if c["kind"] == "linear":
        size = 1 if c["dtype"] == "i8" else 2
        b, by, fl = c["batch"], 0, 0
        for _, n, k in _linear_shapes(c):
            by += n * k * size + 2 * b * (n + k) + (2 * n if size == 1 else 0)
            fl += 2 * b * n * k
        return {"bytes": by, "flops": fl}
    q, ctx = _lengths(c)
    tokens, pairs = sum(q), sum(x * y + x * (x + 1) // 2 for x, y in zip(q, ctx))
    kv = 4 * (tokens + sum(ctx)) * c["kv_heads"] * c["head"]
    by = kv + 4 * tokens * c["heads"] * c["head"]
    fl = 4 * pairs * c["heads"] * c["head"]
    if c["kind"] == "block":
        attn, kvd = c["heads"] * c["head"], 2 * c["kv_heads"] * c["head"]
        by += 2 * c["hidden"] * (2 * attn + kvd) + 2 * c["batch"] * (6 * c["hidden"] + 4 * attn + 2 * kvd)
        fl += 2 * c["batch"] * c["hidden"] * (2 * attn + kvd)
    return {"bytes": by, "flops": fl}


def tolerance(c):
    """About four times the distance from exact() measured on the kinds below:
    one rounding of the result for norms, rotary, convolution and weight
    products, probabilities rounded to 16 bits for attention, and a chain of
    such roundings for the decode block."""
    bf16 = c.get("dtype") == "bf16"
    if c["kind"] in ("tokens", "conv", "linear"):
        return {"rel": 8e-3 if bf16 else 1e-3}
    if c["kind"] == "attn":
        return {"rel": 1e-2 if bf16 else 1.2e-3}
    return {"rel": 1.6e-2 if bf16 else 2e-3}


# ------------------------------------------------------------------- inputs

class _Rand:
    def __init__(self, seed):
        self.g = torch.Generator(device="cuda").manual_seed(int(seed))

    def normal(self, *shape, scale=1.0, dtype=torch.float16):
        out = torch.empty(shape, dtype=dtype, device="cuda")
        flat = out.view(-1)
        for i in range(0, flat.numel(), 1 << 27):  # bounds the 32-bit intermediate
            part = flat[i:i + (1 << 27)]
            part.copy_(torch.randn(part.numel(), generator=self.g, device="cuda").mul_(scale))
        return out

    def uniform(self, n, lo, hi, dtype=torch.float16):
        u = torch.rand(n, generator=self.g, device="cuda")
        return (u * (hi - lo) + lo).to(dtype)

    def int8(self, *shape):
        return torch.randint(-127, 128, shape, generator=self.g, device="cuda", dtype=torch.int8)

    def perm(self, n):
        return torch.randperm(n, generator=self.g, device="cuda")


def _i32(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


def _cumulative(lengths):
    out = [0]
    for n in lengths:
        out.append(out[-1] + n)
    return _i32(out)


def _paged(r, c, kv_lens, dt):
    """Paged caches of the sequences' pages in a shuffled order, with the
    block table that leads to them."""
    pages = [(n + c["block"] - 1) // c["block"] for n in kv_lens]
    perm = r.perm(sum(pages)).int()
    table = torch.zeros(len(pages), max(pages), dtype=torch.int32, device="cuda")
    at = 0
    for i, n in enumerate(pages):
        table[i, :n] = perm[at:at + n]
        at += n
    shape = (at, c["kv_heads"], c["block"], c["head"])
    return r.normal(*shape, dtype=dt), r.normal(*shape, dtype=dt), table


def _angles(positions, dim):
    """float32 [max_position, dim] cos then sin, as a model keeps it."""
    inv = 10000.0 ** (-torch.arange(0, dim, 2, dtype=torch.float64, device="cuda") / dim)
    a = torch.arange(positions, dtype=torch.float64, device="cuda")[:, None] * inv
    return torch.cat([a.cos(), a.sin()], 1).float()


def prepare(c, seed):
    r = _Rand(seed)
    s = {"case": c}
    return {"tokens": _prepare_tokens, "conv": _prepare_conv, "linear": _prepare_linear,
            "attn": _prepare_attn, "block": _prepare_block}[c["kind"]](c, r, s)


def _prepare_tokens(c, r, s):
    dt, t, hid = DTYPES[c["dtype"]], c["tokens"], c["hidden"]
    pages = max(8, (2 * t + c["block"] - 1) // c["block"])
    cache = (pages, c["kv_heads"], c["block"], c["head"])
    s.update(
        x=r.normal(t, hid, dtype=dt), residual=r.normal(t, hid, dtype=dt),
        weight=r.uniform(hid, 0.5, 1.5, dt), out=torch.empty(t, hid, dtype=dt, device="cuda"),
        residual_out=torch.empty(t, hid, dtype=dt, device="cuda"),
        positions=(torch.arange(t, device="cuda") * 7 + c["lens"]) % 4096,
        q=r.normal(t, c["heads"], c["head"], dtype=dt),
        k=r.normal(t, c["kv_heads"], c["head"], dtype=dt),
        v=r.normal(t, c["kv_heads"], c["head"], dtype=dt),
        slots=r.perm(pages * c["block"])[:t].contiguous(),
        kc=torch.zeros(cache, dtype=dt, device="cuda"),
        vc=torch.zeros(cache, dtype=dt, device="cuda"), angles=_angles(4096, c["head"]))
    return s


def _prepare_conv(c, r, s):
    n, _ = _lengths(c)
    dim, total, w = c["dim"], sum(n), c["width"]
    if c["layout"] == "rows":
        x = r.normal(dim, total)
        out = torch.empty_like(x)
    else:  # the transposed view of token-major activations
        x = r.normal(total, dim).t()
        out = torch.empty(total, dim, dtype=torch.float16, device="cuda").t()
    has_state = [i % 2 for i in range(c["batch"])]
    s.update(x=x, out=out, weight=r.normal(w, dim, scale=0.5),
             state=r.normal(c["batch"] + 2, w - 1, dim), starts=_cumulative(n),
             entries=r.perm(c["batch"] + 2)[:c["batch"]].int(),
             has_state=torch.tensor(has_state, dtype=torch.int8, device="cuda"))
    return s


def _prepare_linear(c, r, s):
    i8 = c["dtype"] == "i8"
    dt = torch.float16 if i8 else DTYPES[c["dtype"]]
    s["parts"] = []
    for _, n, k in _linear_shapes(c):
        x, y = r.normal(c["batch"], k, dtype=dt), torch.empty(c["batch"], n, dtype=dt, device="cuda")
        if i8:
            s["parts"].append((r.int8(n, k), r.uniform(n, 0.001, 0.01), x, y))
        else:
            s["parts"].append((r.normal(n, k, scale=0.02, dtype=dt), None, x, y))
    return s


def _prepare_attn(c, r, s):
    dt = DTYPES[c["dtype"]]
    q, ctx = _lengths(c)
    kv = [a + b for a, b in zip(q, ctx)]
    kc, vc, table = _paged(r, c, kv, dt)
    qt = r.normal(sum(q), c["heads"], c["head"], dtype=dt)
    s.update(q=qt, kc=kc, vc=vc, table=table, out=torch.empty_like(qt), starts=_cumulative(q),
             kv_lens=_i32(kv), max_q=max(q), max_kv=max(kv), scale=1.0 / math.sqrt(c["head"]))
    return s


def _prepare_block(c, r, s):
    dt, b, hid = DTYPES[c["dtype"]], c["batch"], c["hidden"]
    attn, kvd = c["heads"] * c["head"], c["kv_heads"] * c["head"]
    _, ctx = _lengths(c)
    kv = [n + 1 for n in ctx]
    kc, vc, table = _paged(r, c, kv, dt)
    last = _i32(ctx).long()
    page = table.gather(1, (last // c["block"])[:, None])[:, 0].long()

    def out(*shape):
        return torch.empty(shape, dtype=dt, device="cuda")

    s.update(
        x=r.normal(b, hid, dtype=dt), residual=r.normal(b, hid, dtype=dt),
        w_in=r.uniform(hid, 0.5, 1.5, dt), w_post=r.uniform(hid, 0.5, 1.5, dt),
        wq=r.normal(attn, hid, scale=hid ** -0.5, dtype=dt),
        wkv=r.normal(2 * kvd, hid, scale=hid ** -0.5, dtype=dt),
        wo=r.normal(hid, attn, scale=attn ** -0.5, dtype=dt),
        kc=kc, vc=vc, table=table, positions=last, slots=page * c["block"] + last % c["block"],
        starts=_cumulative([1] * b), kv_lens=_i32(kv), max_kv=max(kv),
        scale=1.0 / math.sqrt(c["head"]), angles=_angles(max(kv), c["head"]),
        h=out(b, hid), h_res=out(b, hid), q=out(b, attn), kv=out(b, 2 * kvd),
        o=out(b, c["heads"], c["head"]), y=out(b, hid), y_norm=out(b, hid), y_res=out(b, hid))
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):  # one eager step before the capture
        _block_step(s)
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        _block_step(s)
    return s


def _block_step(s):
    c, ops = s["case"], torch.ops.tecoops
    b, d, kvd = c["batch"], c["head"], c["kv_heads"] * c["head"]
    ops.rms_norm(s["x"], s["w_in"], s["residual"], s["h"], s["h_res"], EPS)
    ops.gemv(s["wq"], s["h"], s["q"])
    ops.gemv(s["wkv"], s["h"], s["kv"])
    ops.rotary_reshape_and_cache(s["positions"], s["q"], s["kv"][:, :kvd], s["kv"][:, kvd:],
                                 s["slots"], s["kc"], s["vc"], d, s["angles"], True, 10000.0, d,
                                 False)
    ops.flash_attn_varlen_func(s["q"].view(b, c["heads"], d), s["kc"], s["vc"], 1, s["starts"],
                               s["max_kv"], None, s["kv_lens"], s["scale"], True, None,
                               s["table"], False, s["o"])
    ops.gemv(s["wo"], s["o"].view(b, c["heads"] * d), s["y"])
    ops.rms_norm(s["y"], s["w_post"], s["h_res"], s["y_norm"], s["y_res"], EPS)


# -------------------------------------------------------------------- one pass

def run(s):
    c = s["case"]
    if c["kind"] == "tokens":
        tecoops.rms_norm(s["x"], s["weight"], s["residual"], s["out"], s["residual_out"], EPS)
        tecoops.rotary_reshape_and_cache(s["positions"], s["q"], s["k"], s["v"], s["slots"],
                                         s["kc"], s["vc"], c["head"], s["angles"], c["neox"])
        return {"out": s["out"], "residual_out": s["residual_out"], "q": s["q"], "kc": s["kc"],
                "vc": s["vc"]}
    if c["kind"] == "conv":
        tecoops.causal_conv1d_fn_torch(s["out"], s["state"], s["x"], s["weight"], s["starts"],
                                       s["entries"], s["has_state"], -1)
        return {"out": s["out"], "state": s["state"]}
    if c["kind"] == "linear":
        for w, scales, x, y in s["parts"]:
            if scales is None:
                tecoops.gemv(w, x, y)
            else:
                tecoops.gemv_int8(w, scales, x, y)
        return [p[3] for p in s["parts"]]
    if c["kind"] == "attn":
        tecoops.flash_attn_varlen_func(s["q"], s["kc"], s["vc"], s["max_q"], s["starts"],
                                       s["max_kv"], None, s["kv_lens"], s["scale"], True, None,
                                       s["table"], False, s["out"])
        return s["out"]
    s["graph"].replay()
    return {k: s[k] for k in ("q", "o", "y_norm", "y_res", "kc", "vc")}


# ------------------------------------------------------------- 64-bit results

def _rms(v, w):
    return v * torch.rsqrt(v.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rotate(x, positions, angles, neox):
    """x [T, heads, D] rotated, with the model's 32-bit angles."""
    half = x.shape[-1] // 2
    a = angles.double()[positions][:, None]
    cos, sin = a[..., :half], a[..., half:]
    if neox:
        x1, x2 = x[..., :half], x[..., half:]
        return torch.cat([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1)
    x1, x2 = x[..., 0::2], x[..., 1::2]
    return torch.stack([x1 * cos - x2 * sin, x2 * cos + x1 * sin], -1).flatten(-2)


def _store(cache, slots, rows, block):
    cache = cache.double()
    cache[slots // block, :, slots % block] = rows
    return cache


def _attention(c, q, kc, vc, table, q_lens, kv_lens, scale):
    """q [tokens, heads, D] in 64 bits over the paged caches."""
    out, at = torch.empty_like(q), 0
    g = c["heads"] // c["kv_heads"]
    for i, (n, m) in enumerate(zip(q_lens, kv_lens)):
        pages = table[i, :(m + c["block"] - 1) // c["block"]].long()
        k = kc[pages].transpose(0, 1).reshape(c["kv_heads"], -1, c["head"])[:, :m].double()
        v = vc[pages].transpose(0, 1).reshape(c["kv_heads"], -1, c["head"])[:, :m].double()
        qi = q[at:at + n].double()
        # the rows that fit about 1 GB of scores at a time
        step = max(1, (1 << 27) // (g * m))
        for r0 in range(0, n, step):
            rows = qi[r0:r0 + step]
            hidden = (torch.arange(m, device="cuda")[None] >
                      torch.arange(r0, r0 + rows.shape[0], device="cuda")[:, None] + (m - n))
            for h in range(c["kv_heads"]):
                x = rows[:, h * g:(h + 1) * g].transpose(0, 1).reshape(-1, c["head"])
                p = (x @ k[h].t().contiguous()).view(g, rows.shape[0], m) * scale
                p = p.masked_fill_(hidden, -math.inf).softmax(-1)
                o = (p.view(-1, m) @ v[h]).view(g, rows.shape[0], c["head"])
                out[at + r0:at + r0 + rows.shape[0], h * g:(h + 1) * g] = o.transpose(0, 1)
        at += n
    return out


def exact(c, seed):
    s = prepare(c, seed)
    if c["kind"] == "tokens":
        v = s["x"].double() + s["residual"].double()
        q = _rotate(s["q"].double(), s["positions"], s["angles"], c["neox"])
        k = _rotate(s["k"].double(), s["positions"], s["angles"], c["neox"])
        return {"out": _rms(v, s["weight"]), "residual_out": v, "q": q,
                "kc": _store(s["kc"], s["slots"], k, c["block"]),
                "vc": _store(s["vc"], s["slots"], s["v"].double(), c["block"])}
    if c["kind"] == "conv":
        w, starts, at = c["width"], s["starts"].tolist(), s["entries"].tolist()
        out = torch.empty(s["x"].shape, dtype=torch.float64, device="cuda")
        state = s["state"].double()
        for i in range(c["batch"]):
            x = s["x"][:, starts[i]:starts[i + 1]].double()
            before = state[at[i]].t() if i % 2 else torch.zeros_like(state[at[i]].t())
            full = torch.cat([before, x], 1)
            y = sum(full[:, j:j + x.shape[1]] * s["weight"][j].double()[:, None] for j in range(w))
            out[:, starts[i]:starts[i + 1]] = y * torch.sigmoid(y)
            state[at[i]] = full[:, full.shape[1] - (w - 1):].t()
        return {"out": out, "state": state}
    if c["kind"] == "linear":
        got = []
        for w, scales, x, _ in s["parts"]:
            y = torch.empty(x.shape[0], w.shape[0], dtype=torch.float64, device="cuda")
            for n in range(0, w.shape[0], 4096):
                y[:, n:n + 4096] = x.double() @ w[n:n + 4096].double().t().contiguous()
            got.append(y if scales is None else y * scales.double())
        return got
    if c["kind"] == "attn":
        q, ctx = _lengths(c)
        return _attention(c, s["q"].double(), s["kc"], s["vc"], s["table"], q,
                          s["kv_lens"].tolist(), s["scale"])
    d, kvd, b = c["head"], c["kv_heads"] * c["head"], c["batch"]
    res = s["x"].double() + s["residual"].double()
    h = _rms(res, s["w_in"])
    q = (h @ s["wq"].double().t().contiguous()).view(b, c["heads"], d)
    kv = h @ s["wkv"].double().t().contiguous()
    q = _rotate(q, s["positions"], s["angles"], True)
    k = _rotate(kv[:, :kvd].reshape(b, c["kv_heads"], d), s["positions"], s["angles"], True)
    kc = _store(s["kc"], s["slots"], k, c["block"])
    vc = _store(s["vc"], s["slots"], kv[:, kvd:].reshape(b, c["kv_heads"], d), c["block"])
    o = _attention(c, q, kc, vc, s["table"], [1] * b, s["kv_lens"].tolist(), s["scale"])
    y_res = o.view(b, -1) @ s["wo"].double().t().contiguous() + res
    return {"q": q.view(b, -1), "o": o, "y_norm": _rms(y_res, s["w_post"]), "y_res": y_res,
            "kc": kc, "vc": vc}
