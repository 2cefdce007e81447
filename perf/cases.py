"""The work this framework is used for, as measurable cases.

Every case goes through the package's public entry points (``PagedKv`` and
``attention``) the way a serving engine or a model's forward calls them.  The
shapes are those of the benchmark configurations (GPT-2: 12 layers x 12 heads
x 64; the long-context shape: 32 heads x 128), with contexts, batch sizes and
prompt lengths over their ranges, odd ones included.

A case names its kind:

* ``resident``: ``decode_steps`` -- several decode steps of a few sequences
  enqueued at once, the single-user generation loop;
* ``step``: ``step`` -- one iteration of continuous batching over every layer
  (decode rows, prompt chunks, speculative verify or whole prompts);
* ``layers``: ``step_begin`` / ``step_layer`` per layer / ``step_end`` -- the
  same iteration as a model's forward runs it;
* ``block``: one layer's QKV projection with the append in its epilogue
  (``qkv_append``), then its paged attention (``attention``);
* ``rows``: ``attention`` over contiguous f32 K/V rows, the CPU engine's op.

Contexts and page orders follow from the case's ``ctx_seed`` (so a case's work
is fixed); every value follows from ``prepare``'s seed.  After a pass that
commits rows, the sequences are truncated back, as a speculative rollback
does, so that a pass can be repeated.
"""
import math
import random

import numpy as np
import torch

import nanoinfer_amd as na
from nanoinfer_amd.batch import w_bytes

GPT2 = dict(n_layer=12, n_head=12, head_dim=64)
LONG = dict(n_layer=1, n_head=32, head_dim=128)


def _paged(kind, shape, seqs, ctx_lo, ctx_hi, new, query, q8=False, chunk=0, split=0, std=1.0, steps=1, ctx_seed=1):
    """seqs sequences of ctx_lo..ctx_hi positions, each appending `new` rows
    and querying the last `query`; `chunk` > 0: one more sequence, appending a
    prompt chunk of that many rows of which the last is queried."""
    return dict(kind=kind, **shape, seqs=seqs, ctx_lo=ctx_lo, ctx_hi=ctx_hi, new=new, query=query, q8=q8, chunk=chunk,
                split=split, std=std, steps=steps, ctx_seed=ctx_seed)


def _block(shape, seqs, ctx_lo, ctx_hi, new, w_format, ctx_seed=1):
    shape = dict(shape, n_layer=1)
    return dict(kind="block", **shape, seqs=seqs, ctx_lo=ctx_lo, ctx_hi=ctx_hi, new=new, query=new, q8=False, chunk=0,
                split=0, std=1.0, steps=1, ctx_seed=ctx_seed, w_format=w_format)


def _rows(n_q, q_pos0, n_head=12, head_dim=64):
    return dict(kind="rows", n_q=n_q, q_pos0=q_pos0, n_head=n_head, head_dim=head_dim)


def listed():
    return [
        # One user generating text: 32 tokens of one sequence in mid-context, the smallest launches there are.
        dict(_paged("resident", GPT2, 1, 517, 517, 1, 1, steps=32), name="generate-1"),
        # Continuous batching in steady state: 63 sequences decode while one more prefills a chunk of its prompt.
        dict(_paged("step", GPT2, 63, 32, 767, 1, 1, chunk=193, ctx_seed=3), name="serve-64"),
        # The same on the int8 cache, which halves the bytes of a context.
        dict(_paged("step", GPT2, 64, 32, 767, 1, 1, q8=True, ctx_seed=4), name="serve-64-q8"),
        # Long-context decode: four 32K-token documents, split into partitions and merged.
        dict(_paged("step", LONG, 4, 32767, 32767, 1, 1, split=512, std=0.5), name="long-4x32k"),
        # Speculative decoding: 32 sequences verify four drafts each.
        dict(_paged("step", GPT2, 32, 128, 1019, 5, 5, ctx_seed=5), name="verify-32x5"),
        # Prompt processing at full load: 16 prompts of 512 tokens, every row attended.
        dict(_paged("step", GPT2, 16, 0, 0, 512, 512), name="prefill-16x512"),
        # A model's forward in steady state: each layer's append and attention is a call of its own.
        dict(_paged("layers", GPT2, 64, 32, 767, 1, 1, ctx_seed=6), name="forward-64"),
        # A model's forward over one user's prompt: the time to the first token.
        dict(_paged("layers", GPT2, 1, 0, 0, 509, 509), name="forward-prompt-509"),
        # One attention layer of a decode batch: projection, append and attention, weights as trained.
        dict(_block(GPT2, 64, 32, 767, 1, "f32", ctx_seed=7), name="layer-64-f32"),
        # One attention layer of two prompts with 4-bit weights, the serving default.
        dict(_block(GPT2, 2, 0, 0, 256, "q4_0"), name="layer-2x256-q4_0"),
        # The CPU engine's op over a full-context prompt, K/V rows contiguous in f32.
        dict(_rows(1024, 0), name="rows-prompt-1024"),
        # The same op for one generated token.
        dict(_rows(1, 1000), name="rows-token-1001"),
    ]


def _log(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi + 0.5)))))))


def draw(rng: random.Random):
    kind = rng.choice(["resident", "serve", "long", "verify", "prompts", "forward", "forward-prompt", "layer",
                       "layer-prompt", "rows-prompt", "rows-token"])
    cs = rng.randrange(1 << 30)
    hi = rng.randint(64, 1000)
    lo = rng.randint(1, hi)
    if kind == "resident":
        return _paged("resident", GPT2, _log(rng, 1, 6), lo, hi, 1, 1, q8=rng.random() < 0.3, steps=rng.randint(4, 8),
                      ctx_seed=cs)
    if kind == "serve":
        chunk = 0 if rng.random() < 0.4 else rng.randint(17, 256)
        return _paged("step", GPT2, _log(rng, 2, 63), min(lo, 700), min(hi, 760), 1, 1, q8=rng.random() < 0.4,
                      chunk=chunk, ctx_seed=cs)
    if kind == "long":
        hi = _log(rng, 2000, 32000)
        return _paged("step", LONG, rng.randint(1, 4), rng.randint(1000, hi), hi, 1, 1,
                      split=rng.choice([0, 0, 512, 1024]), std=0.5, ctx_seed=cs)
    if kind == "verify":
        k = rng.randint(2, 9)
        return _paged("step", GPT2, _log(rng, 1, 32), lo, hi, k, k, q8=rng.random() < 0.3, ctx_seed=cs)
    if kind == "prompts":
        n = _log(rng, 17, 512)
        ctx = 0 if rng.random() < 0.6 else rng.randint(1, 200)
        return _paged("step", GPT2, rng.randint(1, 6), ctx, ctx, n, n, q8=rng.random() < 0.3, ctx_seed=cs)
    if kind == "forward":
        return _paged("layers", GPT2, _log(rng, 2, 64), min(lo, 700), min(hi, 760), 1, 1, q8=rng.random() < 0.3,
                      ctx_seed=cs)
    if kind == "forward-prompt":
        n = _log(rng, 17, 700)
        return _paged("layers", GPT2, rng.randint(1, 3), 0, 0, n, n, q8=rng.random() < 0.3, ctx_seed=cs)
    fmt = rng.choice(["f32", "f16", "q8_0", "q4_0"])
    if kind == "layer":
        return _block(GPT2, _log(rng, 1, 64), min(lo, 700), min(hi, 760), 1, fmt, ctx_seed=cs)
    if kind == "layer-prompt":
        return _block(GPT2, rng.randint(1, 3), 0, 0, _log(rng, 17, 400), fmt, ctx_seed=cs)
    n_head, head_dim = rng.choice([(12, 64), (16, 64), (32, 128)])
    if kind == "rows-prompt":
        n_q = _log(rng, 2, 600 if head_dim == 64 else 250)
        return _rows(n_q, 0 if rng.random() < 0.6 else rng.randint(1, 200), n_head, head_dim)
    return _rows(1, _log(rng, 16, 4000), n_head, head_dim)


# ------------------------------------------------------------------- shapes


def _contexts(case):
    rng = random.Random(case["ctx_seed"])
    ctx = [rng.randint(case["ctx_lo"], case["ctx_hi"]) for _ in range(case["seqs"])]
    if case["chunk"]:  # the prefilling sequence is somewhere in its prompt
        ctx.append(rng.randint(0, 256))
    return ctx


def _work(case):
    """(context, rows appended, rows queried) of each sequence in one step."""
    ctx = _contexts(case)
    work = [(c, case["new"], case["query"]) for c in ctx]
    if case["chunk"]:
        work[-1] = (ctx[-1], case["chunk"], 1)
    return work


def _gen(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _normal(g, shape, std=1.0):
    return torch.randn(shape, generator=g, device="cuda", dtype=torch.float32) * std


def _context_kv(case, g):
    """K and V [n_layer, ctx, C] of each sequence, as its earlier steps appended them."""
    c = case["n_head"] * case["head_dim"]
    for ctx in _contexts(case):
        yield _normal(g, (case["n_layer"], ctx, c), case["std"]), _normal(g, (case["n_layer"], ctx, c), case["std"])


def _step_inputs(case, g):
    n = sum(w[1] for w in _work(case))
    shape = (case["n_layer"], n, case["n_head"] * case["head_dim"])
    if case["kind"] == "resident":
        shape = (case["steps"],) + shape
    return _normal(g, shape), _normal(g, shape, case["std"]), _normal(g, shape, case["std"])


def _weights(case, g):
    """W [3C, C] in the case's format and as the f32 matrix it stands for, and the bias."""
    c = case["n_head"] * case["head_dim"]
    w = _normal(g, (3 * c, c), 1.0 / math.sqrt(c))
    bias = _normal(g, (3 * c,), 0.1)
    fmt, n = case["w_format"], 3 * c * c
    if fmt == "f32":
        return w, w, bias
    if fmt == "f16":
        h = w.half()
        return h.view(torch.uint8).reshape(-1), h.float(), bias
    blocks = w.reshape(-1, 32)
    if fmt == "q8_0":
        d = (blocks.abs().amax(1, keepdim=True) / 127).half()
        q = torch.round(blocks / d.float()).clamp(-127, 127)
        quants = q.to(torch.int8).view(torch.uint8).reshape(-1)
    else:
        d = (blocks.abs().amax(1, keepdim=True) / 8).half()
        q = torch.round(blocks / d.float()).clamp(-8, 7)
        u = (q + 8).to(torch.uint8)
        quants = (u[:, :16] | (u[:, 16:] << 4)).reshape(-1)
    raw = torch.cat([quants, d.reshape(-1).view(torch.uint8)]).contiguous()
    assert raw.numel() == w_bytes(fmt, n)
    return raw, (q * d.float()).reshape(3 * c, c), bias


# ------------------------------------------------------------------ prepare


def _cache(case, g, work):
    """A PagedKv holding the sequences' contexts."""
    steps = case["steps"]
    need = [-(-(ctx + new * steps) // na.KV_BLOCK) for ctx, new, _ in work]
    pages = sum(need) + 8
    order = list(range(pages))
    random.Random(case["ctx_seed"] + 1).shuffle(order)
    kv = na.PagedKv(na.BatchOpts(n_layer=case["n_layer"], n_head=case["n_head"], head_dim=case["head_dim"],
                                 kv_blocks=pages, max_seqs=len(work), n_ctx=max(c + n * steps for c, n, _ in work),
                                 max_rows=max(max(c for c, _, _ in work), sum(n for _, n, _ in work)),
                                 page_order=order, q8=case["q8"]))
    seqs = [kv.add_seq() for _ in work]
    for s, (k, v) in zip(seqs, _context_kv(case, g)):
        n = k.shape[1]
        if n:
            kv.reserve(s, n)
            kv.append(np.stack([np.full(n, s), np.arange(n)], 1), k, v)
            kv.commit(s, n)
    kv.sync()
    return kv, seqs


def prepare(case, seed):
    g = _gen(seed)
    if case["kind"] == "rows":
        # q, k and v are views of the projection's fused [rows][3C] buffer, as the engine keeps them.
        c = case["n_head"] * case["head_dim"]
        n = case["q_pos0"] + case["n_q"]
        qkv = _normal(g, (n, 3 * c))
        return dict(case=case, q=qkv[case["q_pos0"]:, :c], k=qkv[:, c:2 * c], v=qkv[:, 2 * c:],
                    out=torch.empty((case["n_q"], c), device="cuda"))
    work = _work(case)
    kv, seqs = _cache(case, g, work)
    state = dict(case=case, kv=kv, seqs=seqs, ctx=[w[0] for w in work])
    if case["kind"] == "block":
        c = case["n_head"] * case["head_dim"]
        rows = np.concatenate([np.stack([np.full(n, s), ctx + np.arange(n)], 1)
                               for s, (ctx, n, _) in zip(seqs, work)]).astype(np.uint32)
        for s, (ctx, n, _) in zip(seqs, work):
            kv.reserve(s, ctx + n)
        raw, _, bias = _weights(case, g)
        x = _normal(g, (len(rows), c))
        state.update(rows=rows, x=x, w=raw, bias=bias, q=torch.empty_like(x), out=torch.empty_like(x))
        return state
    q, k, v = _step_inputs(case, g)
    out = torch.zeros_like(q)
    state.update(q=q, k=k, v=v, out=out,
                 work=np.array([(s, n, nq) for s, (_, n, nq) in zip(seqs, work)], dtype=np.uint32))
    if case["kind"] == "layers":
        state["layers"] = [(q[l], k[l], v[l], out[l]) for l in range(case["n_layer"])]
    return state


# ---------------------------------------------------------------------- run


def _rollback(s):
    kv = s["kv"]
    for seq, ctx in zip(reversed(s["seqs"]), reversed(s["ctx"])):
        kv.truncate(seq, ctx)


def run(s):
    case = s["case"]
    kind = case["kind"]
    if kind == "rows":
        return na.attention(s["q"], s["k"], s["v"], case["n_q"], case["q_pos0"], case["n_head"], case["head_dim"],
                            out=s["out"])
    kv = s["kv"]
    if kind == "block":
        q = kv.qkv_append(s["rows"], s["x"], s["w"], s["bias"], q_out=s["q"], layer=0, w_format=case["w_format"])
        return {"q": q, "out": kv.attention(q, s["rows"], out=s["out"], layer=0)}
    if kind == "resident":
        out = kv.decode_steps(s["seqs"], s["q"], s["k"], s["v"], out=s["out"], split_tokens=case["split"])
    elif kind == "step":
        out = kv.step(s["work"], s["q"], s["k"], s["v"], out=s["out"], split_tokens=case["split"])
    else:
        kv.step_begin(s["work"], split_tokens=case["split"])
        for l, (q, k, v, o) in enumerate(s["layers"]):
            kv.step_layer(l, q, k, v, out=o)
        kv.step_end()
        out = s["out"]
    _rollback(s)
    return out


# --------------------------------------------------------------------- work


def work(case):
    h, d = case["n_head"], case["head_dim"]
    c = h * d
    if case["kind"] == "rows":
        n_kv = case["q_pos0"] + case["n_q"]
        keys = case["n_q"] * case["q_pos0"] + case["n_q"] * (case["n_q"] + 1) // 2
        return {"bytes": 4 * c * (2 * case["n_q"] + 2 * n_kv), "flops": 4 * c * keys}
    # bytes of one cached position (K and V of a layer), and of an appended row's f32 input
    pos = 2 * h * (d + 4) if case["q8"] else 4 * c
    nbytes, flops, rows = 0, 0, 0
    for ctx, n, nq in _work(case):
        for t in range(case["steps"]):
            end = ctx + (t + 1) * n
            first = end - nq  # position of the first queried row
            keys = nq * first + nq * (nq + 1) // 2
            rows += n
            nbytes += n * pos + nq * 8 * c + (end * pos + -(-end // na.KV_BLOCK) * 4)
            if case["kind"] != "block":
                nbytes += n * 8 * c
            flops += 4 * c * keys
    nbytes, flops = nbytes * case["n_layer"], flops * case["n_layer"]
    if case["kind"] == "block":
        # x read; q written once more by the projection (its read is counted above)
        nbytes += rows * 8 * c + w_bytes(case["w_format"], 3 * c * c) + 12 * c
        flops += 2 * rows * 3 * c * c
    return {"bytes": nbytes, "flops": flops}


def tolerance(case):
    if case["kind"] == "block":
        # K/V are rounded to f16 from sums in 32 bits: a sum in another order
        # rounds a few of them to the neighbouring f16 (1e-5 measured against
        # 64 bits; one value by up to its f16 spacing).
        return {"rel": 4e-5, "max": 2e-3}
    # About ten times the error against 64 bits (1e-7 to 3e-7 measured).
    return {"rel": 4e-6, "max": 2e-4}


# -------------------------------------------------------------------- exact


def _attend(q, k, v, pos0, h, d):
    """Causal attention in 64 bits: q [L, nq, C] at positions pos0.. over k, v [L, n, C]."""
    n_lay, nq, c = q.shape
    n = k.shape[1]
    out = torch.empty((n_lay, nq, c), dtype=torch.float64, device=q.device)
    hidden = torch.arange(n, device=q.device)[None, :] > (pos0 + torch.arange(nq, device=q.device))[:, None]
    for l in range(n_lay):
        qh = q[l].double().reshape(nq, h, d).transpose(0, 1).contiguous()
        kh = k[l].double().reshape(n, h, d).permute(1, 2, 0).contiguous()
        vh = v[l].double().reshape(n, h, d).transpose(0, 1).contiguous()
        s = torch.matmul(qh, kh) / math.sqrt(d)
        s.masked_fill_(hidden, -math.inf)
        out[l] = torch.matmul(torch.softmax(s, -1), vh).transpose(0, 1).reshape(nq, c)
    return out


def _stored(x, case):
    """The values the cache holds of f32 rows x [L, n, C]."""
    if not case["q8"]:
        return x.half().double()
    b = x.reshape(x.shape[0], x.shape[1], case["n_head"], case["head_dim"])
    # Correctly rounded f32 quotients (torch divides by a scalar through its reciprocal).
    scale = (b.abs().amax(-1, keepdim=True).double() / 127).float()
    inv = torch.where(scale > 0, 1 / scale.double(), torch.zeros_like(scale).double()).float()
    return (torch.round(b * inv).clamp(-127, 127).double() * scale.double()).reshape(x.shape)


def exact(case, seed):
    g = _gen(seed)
    h, d = case["n_head"], case["head_dim"]
    c = h * d
    if case["kind"] == "rows":
        n = case["q_pos0"] + case["n_q"]
        qkv = _normal(g, (n, 3 * c))
        return _attend(qkv[None, case["q_pos0"]:, :c], qkv[None, :, c:2 * c], qkv[None, :, 2 * c:], case["q_pos0"], h,
                       d)[0]
    ctx_kv = [(_stored(k, case), _stored(v, case)) for k, v in _context_kv(case, g)]
    work = _work(case)
    if case["kind"] == "block":
        _, w, bias = _weights(case, g)
        x = _normal(g, (sum(n for _, n, _ in work), c))
        y = torch.matmul(x.double(), w.double().t().contiguous()) + bias.double()
        q, k, v = (t.contiguous()[None] for t in y.split(c, 1))
        out = torch.empty_like(q)
    else:
        q, k, v = _step_inputs(case, g)
        out = torch.zeros(q.shape, dtype=torch.float64, device="cuda")
    row = 0
    for i, ((ctx, n, nq), (ck, cv)) in enumerate(zip(work, ctx_kv)):
        if case["kind"] == "resident":
            for t in range(case["steps"]):
                ck = torch.cat([ck, _stored(k[t, :, i:i + 1], case)], 1)
                cv = torch.cat([cv, _stored(v[t, :, i:i + 1], case)], 1)
                out[t, :, i:i + 1] = _attend(q[t, :, i:i + 1], ck, cv, ctx + t, h, d)
            continue
        kk = torch.cat([ck, _stored(k[:, row:row + n], case)], 1)
        vv = torch.cat([cv, _stored(v[:, row:row + n], case)], 1)
        last = slice(row + n - nq, row + n)
        out[:, last] = _attend(q[:, last], kk, vv, ctx + n - nq, h, d)
        row += n
    return {"q": q[0], "out": out[0]} if case["kind"] == "block" else out
