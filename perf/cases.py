"""Timed workloads of the session attention path, through the package's public
entry points (toklet_amd.ops, toklet_amd.kv, toklet_amd.session).

A case is a dict of plain values: "op" names the call sequence, the rest its
sizes.  listed() holds the representative ones, draw() gives others of the same
ranges, prepare() makes what a program has in hand before the call, run() is one
pass, and exact() is the same result in 64-bit floating point from plain torch,
with the operands rounded to the storage dtype the call is asked to use.
"""

from __future__ import annotations

import math

import torch

from toklet_amd import kv, ops, session

_DT = {"f32": torch.float32, "f16": torch.float16, "bf16": torch.bfloat16}
_ES = {"f32": 4, "f16": 2, "bf16": 2}
# Query heads / KV heads / head_dim of the models the path serves.
_QWEN2, _QWEN3, _LLAMA3, _GEMMA3 = (14, 2, 64), (16, 8, 128), (32, 8, 128), (8, 4, 256)
_SHAPES = (_QWEN2, _QWEN3, _LLAMA3, _GEMMA3)


def listed():
    return [
        # One decode step of a short chat: append the token's K/V, attend.  A few
        # hundred keys, so launches and latency are all of it.
        dict(name="step_bf16", op="append", tokens=1, hq=16, hkv=8, d=128, offset=300, dtype="bf16", queued=True),
        # One layer of a 128-token prompt chunk near the end of a 2048-token
        # prompt: RMSNorm, rotary, append and attention.
        dict(name="chunk_bf16", op="produce", tokens=128, hq=16, hkv=8, d=128, offset=1920, dtype="bf16", queued=True),
        # The same chunk at the FP32 shape, whose caches keep FP32 rows.
        dict(name="chunk_f32", op="append", tokens=128, hq=14, hkv=2, d=64, offset=1920, dtype="f32", queued=True),
        # A 512-token FP32 prompt in one full-prefix call, waited for as the
        # reference operator is.
        dict(name="prefill_f32", op="attention", tokens=512, hq=14, hkv=2, d=64, dtype="f32", diag=False, queued=False),
        # Full-prefix attention with the score and probability matrices the
        # reference operators return, at an odd length.
        dict(name="diagnostics_bf16", op="attention", tokens=300, hq=16, hkv=8, d=128, dtype="bf16", diag=True, queued=False),
        # A serving batch: 64 sessions of mixed lengths, one new token each.
        dict(name="decode_batch", op="decode_batch", batch=64, shortest=512, longest=8192, hq=16, hkv=8, d=128,
             dtype="f16", queued=True),
        # A serving batch: 32 cached prompts of 4096 tokens, 128 new tokens each.
        dict(name="prefill_batch", op="prefill_batch", batch=32, tokens=128, cached=4096, hq=32, hkv=8, d=128,
             dtype="bf16", queued=True),
        # A sliding layer's chunk over a wrapped ring: prepare, view, attention
        # over its spans, score softcap.
        dict(name="ring_chunk", op="ring", tokens=128, committed=3000, window=1024, hq=8, hkv=4, d=256, dtype="bf16",
             softcap=50.0, queued=True),
        # A chunk of a global layer with 512-wide heads and one KV head.
        dict(name="window_512", op="window", tokens=128, keys=1025, window=0, hq=8, hkv=1, d=512, dtype="bf16",
             softcap=0.0, queued=False),
        # The step after attention: one row's logits over the vocabulary and its
        # greedy token.
        dict(name="project_row", op="project", rows=1, hidden=896, vocab=151936, queued=True),
        # The final logits' softcap over a large vocabulary, in place.
        dict(name="softcap", op="softcap", n=262144, cap=30.0, queued=True),
        # A whole request: six layers (five sliding, one global), a prompt in
        # 128-token chunks, then single-token steps.
        dict(name="session", op="session", prompt=2050, steps=33, window=1024, hq=8, hkv=4, d=256, dtype="bf16",
             softcap=50.0, queued=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choice(("append", "append", "produce", "attention", "decode_batch", "prefill_batch", "ring", "window",
                     "project", "softcap", "session"))
    hq, hkv, d = rng.choice(_SHAPES)
    c = dict(op=op, hq=hq, hkv=hkv, d=d, dtype=rng.choice(("bf16", "bf16", "f16", "f32")), queued=rng.random() < 0.6)
    if op in ("append", "produce"):
        c.update(tokens=rng.choice((1, _log(rng, 2, 512))), offset=_log(rng, 1, 8192))
        if c["dtype"] == "f32":
            c.update(offset=_log(rng, 1, 4096))
    elif op == "attention":
        c.update(tokens=_log(rng, 5, 1024), diag=rng.random() < 0.4)
    elif op == "decode_batch":
        longest = _log(rng, 64, 8192)
        c.update(batch=_log(rng, 2, 64), shortest=max(1, longest // rng.choice((1, 4, 16))), longest=longest,
                 dtype=rng.choice(("bf16", "f16")))
        if d == 256:
            c.update(batch=min(c["batch"], 32))
    elif op == "prefill_batch":
        c.update(batch=_log(rng, 2, 24), tokens=_log(rng, 9, 128), cached=_log(rng, 16, 4096),
                 dtype=rng.choice(("bf16", "f16")))
    elif op == "ring":
        w = _log(rng, 64, 1024)
        c.update(tokens=_log(rng, 1, 200), window=w, committed=_log(rng, 1, 4 * w), softcap=rng.choice((0.0, 50.0)))
    elif op == "window":
        t = _log(rng, 1, 256)
        c.update(tokens=t, keys=t + _log(rng, 1, 2048), window=rng.choice((0, _log(rng, 16, 1024))),
                 softcap=rng.choice((0.0, 30.0, 50.0)))
        if rng.random() < 0.4:
            c.update(hq=8, hkv=rng.choice((1, 2)), d=512)
    elif op == "project":
        c = dict(op=op, queued=c["queued"], rows=rng.choice((1, _log(rng, 2, 128))), hidden=hq * d // rng.choice((1, 2)),
                 vocab=_log(rng, 1500, 30000))
    elif op == "softcap":
        c = dict(op=op, queued=c["queued"], n=_log(rng, 500, 1 << 21), cap=rng.choice((30.0, 50.0)))
    else:
        c.update(prompt=_log(rng, 20, 1400), steps=_log(rng, 1, 24), window=_log(rng, 64, 1024),
                 softcap=rng.choice((0.0, 50.0)) if d == 256 else 0.0, dtype=rng.choice(("bf16", "f16")))
    return c


# ---- inputs: N(0, 1) activations, as the path's own tests and benchmark draw them

def _randn(g, *shape):
    return torch.randn(*shape, generator=g, device="cuda")


def _inputs(case, seed):
    g = torch.Generator(device="cuda").manual_seed(seed)
    op, s = case["op"], {}
    dt = _DT.get(case.get("dtype"), torch.float32)
    if op == "project":
        s["x"] = _randn(g, case["rows"], case["hidden"])
        s["w"] = _randn(g, case["vocab"], case["hidden"]) / math.sqrt(case["hidden"])
        return s
    if op == "softcap":
        s["x"] = _randn(g, case["n"]) * 20.0
        return s
    hq, hkv, d = case["hq"], case["hkv"], case["d"]
    if op in ("append", "produce"):
        t, off = case["tokens"], case["offset"]
        s["kc"] = _randn(g, hkv, off + t, d).to(dt)
        s["vc"] = _randn(g, hkv, off + t, d).to(dt)
        s["kp"], s["vp"] = _randn(g, t, hkv, d), _randn(g, t, hkv, d)
        s["qp"] = _randn(g, t, hq, d)
        s["wq"], s["wk"] = 1.0 + 0.02 * _randn(g, d), 1.0 + 0.02 * _randn(g, d)
    elif op == "attention":
        t = case["tokens"]
        s["q"], s["k"], s["v"] = (_randn(g, t, h, d).to(dt) for h in (hq, hkv, hkv))
    elif op in ("decode_batch", "prefill_batch"):
        # Peaky rows: a scale per (session, KV head) for decode, 5% of the key rows
        # eight times larger for prefill.
        cpu = torch.Generator().manual_seed(seed)
        b = case["batch"]
        if op == "decode_batch":
            n = torch.randint(case["shortest"], case["longest"] + 1, (b,), generator=cpu).tolist()
            t = 1
        else:
            n, t = [case["cached"] + case["tokens"]] * b, case["tokens"]
        s["lengths"], s["offsets"] = n, [sum(n[:i]) * hkv * d for i in range(b)]
        total = sum(n) * hkv * d
        s["k"] = torch.randn(total, generator=g, device="cuda", dtype=dt)
        s["v"] = torch.randn(total, generator=g, device="cuda", dtype=dt)
        s["q"] = _randn(g, b, t, hq, d).to(dt)
        if op == "decode_batch":
            scale = torch.empty(b, hkv, device="cuda").uniform_(0.5, 2.0, generator=g)
            for i, o in enumerate(s["offsets"]):
                m = hkv * n[i] * d
                for x in (s["k"], s["v"]):
                    x[o:o + m].view(hkv, n[i] * d).mul_(scale[i][:, None].to(dt))
            s["q"].mul_(scale.repeat_interleave(hq // hkv, 1)[:, None, :, None].to(dt))
        else:
            rows = s["k"].view(-1, d)
            rows.mul_(1.0 + 7.0 * (torch.rand(rows.shape[0], 1, generator=g, device="cuda") < 0.05).to(dt))
    elif op == "ring":
        n, t = case["committed"], case["tokens"]
        s["k"], s["v"] = _randn(g, hkv, n + t, d).to(dt), _randn(g, hkv, n + t, d).to(dt)
        s["q"] = _randn(g, t, hq, d).to(dt)
    elif op == "window":
        s["q"] = _randn(g, case["tokens"], hq, d).to(dt)
        s["k"], s["v"] = (_randn(g, hkv, case["keys"], d).to(dt) for _ in range(2))
    else:
        total = case["prompt"] + case["steps"]
        s["layers"] = [tuple(_randn(g, total, h, d) for h in (hq, hkv, hkv)) for _ in range(6)]
    return s


def prepare(case, seed):
    s = _inputs(case, seed)
    op = case["op"]
    ctx = s["ctx"] = ops.Context(0, synchronous=not case["queued"])
    s["case"] = case
    if op == "project":
        s["tokens"] = torch.zeros(case["rows"], dtype=torch.int32, device="cuda")
        s["logits"] = torch.zeros(case["rows"], case["vocab"], device="cuda")
        return s
    if op == "softcap":
        s["raw"] = s["x"].clone()
        return s
    hq, hkv, d, dt = case["hq"], case["hkv"], case["d"], _DT[case["dtype"]]
    if op != "session":
        rows = {"decode_batch": case.get("batch", 0), "prefill_batch": case.get("batch", 0) * case.get("tokens", 0)}
        s["out"] = torch.zeros(rows.get(op, case.get("tokens", 0)) * hq * d, device="cuda")
    if op in ("append", "produce"):
        t, off = case["tokens"], case["offset"]
        if op == "append":
            owner = s["owner"] = kv.LayerKv(ctx, hkv, d, off + t, dt)
            s["k"], s["v"] = owner.committed()
            for view, rows in ((s["k"], s["kc"]), (s["v"], s["vc"])):
                view.copy_(rows)
                view.owner = owner  # the owner's memory lives as long as a view of it
        else:
            s["k"], s["v"] = s["kc"], s["vc"]
        del s["kc"], s["vc"]
        s["q"] = s["qp"].to(dt)
        s["shape"] = ops.CachedAttentionShape(t, hq, hkv, d, off + t, off)
        s["producer"] = ops.ProducerShape(t, hq, hkv, d, off, theta=1e6)
    elif op == "attention":
        t = case["tokens"]
        s["scores"] = torch.zeros(hq * t * t, device="cuda") if case["diag"] else None
        s["probs"] = torch.zeros(hq * t * t, device="cuda") if case["diag"] else None
        s["shape"] = ops.AttentionShape(t, hq, hkv, d)
    elif op in ("decode_batch", "prefill_batch"):
        s["strides"] = [n * d for n in s["lengths"]]
        s["positions"] = [n - case.get("tokens", 1) for n in s["lengths"]]
    elif op == "ring":
        n, t, w = case["committed"], case["tokens"], case["window"]
        ring = s["owner"] = kv.WindowKvCache(ctx, hkv, d, w, max(w, n + t), w, dt)
        for a in range(0, n, w):  # the history, committed window by window
            b = min(n, a + w)
            rows = [x[:, a:b].contiguous() for x in (s["k"], s["v"])]
            ring.commit(ring.prepare(rows[0], rows[1], b - a))
            ctx.synchronize()
        s["kn"], s["vn"] = s["k"][:, n:].contiguous(), s["v"][:, n:].contiguous()
        del s["k"], s["v"]
    elif op == "window":
        t, n = case["tokens"], case["keys"]
        s["shape"] = ops.WindowAttentionShape(t, n, n, hq, hkv, d, n - t, 0, case["window"] or None, 1.0 / math.sqrt(d),
                                              case["softcap"])
    else:
        total = case["prompt"] + case["steps"]
        s["outs"] = [torch.zeros(total, hq * d, device="cuda") for _ in s["layers"]]
        s["io"] = [session.LayerIo(q, k, v, o) for (q, k, v), o in zip(s["layers"], s["outs"])]
        s["session"] = session.Session(ctx, session.Options(
            capacity=total, prefill_chunk_size=128, vocab_size=262144, layers=6, query_heads=hq, kv_heads=hkv, head_dim=d,
            storage=case["dtype"], score_scale=1.0 / math.sqrt(d), softcap=case["softcap"], theta=1e6,
            layer_windows=[case["window"]] * 5 + [0]))
        s["ids"] = [1] * total
    return s


def run(s):
    c, ctx = s["case"], s["ctx"]
    op = c["op"]
    if op == "append":
        s["owner"].append(s["kp"], s["vp"], c["offset"])
        ops.attention_cached(ctx, s["q"], s["k"], s["v"], s["out"], None, None, s["shape"])
        return {"context": s["out"], "k": s["k"], "v": s["v"]}
    if op == "produce":
        ops.produce_qkv(ctx, s["producer"], s["qp"], s["kp"], s["vp"], s["wq"], s["wk"], s["q"],
                        s["k"][:, c["offset"]:], s["v"][:, c["offset"]:], (c["offset"] + c["tokens"]) * c["d"])
        ops.attention_cached(ctx, s["q"], s["k"], s["v"], s["out"], None, None, s["shape"])
        return {"context": s["out"], "k": s["k"], "v": s["v"], "q": s["q"]}
    if op == "attention":
        ops.attention(ctx, s["q"], s["k"], s["v"], s["out"], s["scores"], s["probs"], s["shape"])
        return {"context": s["out"], "scores": s["scores"], "probs": s["probs"]}
    if op == "decode_batch":
        ops.decode_batch(ctx, s["q"], s["k"], s["v"], s["offsets"], s["strides"], s["lengths"], s["out"],
                         query_heads=c["hq"], kv_heads=c["hkv"], head_dim=c["d"], scale=1.0 / math.sqrt(c["d"]))
        return {"context": s["out"]}
    if op == "prefill_batch":
        ops.prefill_batch(ctx, s["q"], s["k"], s["v"], s["offsets"], s["strides"], s["positions"], s["out"],
                          tokens=c["tokens"], query_heads=c["hq"], kv_heads=c["hkv"], head_dim=c["d"],
                          scale=1.0 / math.sqrt(c["d"]))
        return {"context": s["out"]}
    if op == "ring":
        view = s["owner"].view(s["owner"].prepare(s["kn"], s["vn"], c["tokens"]))
        shape = view.attention_shape(c["hq"], 1.0 / math.sqrt(c["d"]))
        shape.softcap = c["softcap"]
        ops.span_attention(ctx, s["q"], view.segments(), s["out"], None, None, shape)
        return {"context": s["out"]}
    if op == "window":
        ops.window_attention(ctx, s["q"], s["k"], s["v"], s["out"], None, None, s["shape"])
        return {"context": s["out"]}
    if op == "project":
        ops.project_greedy(ctx, s["x"], s["w"], s["tokens"], s["logits"])
        return {"tokens": s["tokens"], "logits": s["logits"]}
    if op == "softcap":
        s["x"].copy_(s["raw"])  # the call works in place: fresh logits first
        ops.logit_softcap(ctx, s["x"], c["cap"])
        return {"logits": s["x"]}
    sess = s["session"]
    sess.reset()
    sess.set_tokens(s["ids"][:c["prompt"]])
    sess.evaluate(s["io"])
    sess.append(s["ids"][c["prompt"]:])
    sess.evaluate(s["io"], chunk_limit=1)
    sess.synchronize()
    return {"layer%d" % i: o for i, o in enumerate(s["outs"])}


# ---- the least work of a pass

def _pairs(queries, first, window=0):
    """Visible (query, key) pairs of `queries` rows from position `first`."""
    if not window:
        return queries * first + queries * (queries + 1) // 2
    return sum(min(p + 1, window) for p in range(first, first + queries))


def work(case):
    op = case["op"]
    if op == "project":
        r, h, v = case["rows"], case["hidden"], case["vocab"]
        return {"bytes": 4.0 * (v * h + r * h + r * v + r), "flops": 2.0 * r * h * v}
    if op == "softcap":
        return {"bytes": 16.0 * case["n"], "flops": 30.0 * case["n"]}
    hq, hkv, d, es = case["hq"], case["hkv"], case["d"], _ES[case["dtype"]]
    t = case.get("tokens", 1)
    io = lambda rows: rows * hq * d * (es + 4.0)  # Q in, context out
    rows = lambda n: 2.0 * n * hkv * d * es  # K and V of n keys
    fl = lambda pairs: 4.0 * hq * d * pairs
    if op in ("append", "produce"):
        n = case["offset"] + t
        new = t * hkv * d * 8.0 + rows(t)  # FP32 rows in, storage rows out
        q = t * hq * d * (4.0 + es) if op == "produce" else 0.0
        return {"bytes": io(t) + rows(n) + new + q, "flops": fl(_pairs(t, case["offset"]))}
    if op == "attention":
        diag = 8.0 * hq * t * t if case["diag"] else 0.0
        return {"bytes": io(t) + rows(t) + diag, "flops": fl(_pairs(t, 0))}
    if op == "decode_batch":
        n = case["batch"] * (case["shortest"] + case["longest"]) / 2
        return {"bytes": io(case["batch"]) + rows(n), "flops": fl(n)}
    if op == "prefill_batch":
        b, n = case["batch"], case["cached"] + t
        return {"bytes": b * (io(t) + rows(n)), "flops": fl(b * _pairs(t, case["cached"]))}
    if op == "ring":
        n = min(case["committed"], case["window"] - 1) + t
        return {"bytes": io(t) + rows(n), "flops": fl(_pairs(t, case["committed"], case["window"]))}
    if op == "window":
        w = case["window"]
        first = case["keys"] - t
        n = min(case["keys"], w + t - 1) if w else case["keys"]
        return {"bytes": io(t) + rows(n), "flops": fl(_pairs(t, first, w))}
    total, p, w = case["prompt"] + case["steps"], case["prompt"], case["window"]
    flops = fl(_pairs(total, 0) + 5 * _pairs(total, 0, w))
    # Each chunk and each step reads its visible keys; the projections are FP32.
    starts = [(a, min(a + 128, p)) for a in range(0, p, 128)] + [(a, a + 1) for a in range(p, total)]
    keys = sum(b + 5 * min(b, w + b - a - 1) for a, b in starts)
    return {"bytes": rows(keys) + 6.0 * total * ((hq + 2 * hkv) * d * 4.0 + hkv * d * 2.0 * es + hq * d * 4.0),
            "flops": flops}


def tolerance(case):
    op = case["op"]
    if op == "project":
        # FP32 dot products of a few thousand terms; a row's two best logits may tie.
        return {"rel": 2e-6, "max": 1e-4, "differ": 0.01}
    if op == "softcap":
        return {"rel": 1e-6, "max": 1e-6}
    if case["dtype"] == "f32":
        return {"rel": 1e-5, "max": 2e-4}
    if op == "session" or op == "produce":
        # A 16-bit operand may round the other way after the norm and the rotary.
        return {"rel": 5e-3, "max": 0.1}
    return {"rel": 2e-3, "max": 0.05}


# ---- the same results in 64-bit floating point

def _attend(q, k, v, first, scale, window=0, softcap=0.0):
    """q [T, Hq, D] at positions first.., k/v [Hkv, N, D] from position 0, all
    float64: context [T, Hq, D], scores and probabilities [Hq, T, N]."""
    t, hq, d = q.shape
    hkv, n, _ = k.shape
    qh = q.transpose(0, 1).reshape(hkv, hq // hkv * t, d).contiguous()
    x = torch.matmul(qh, k.transpose(1, 2).contiguous()).reshape(hq, t, n) * scale
    if softcap:
        x = softcap * torch.tanh(x / softcap)
    pos = torch.arange(first, first + t, device=q.device)[:, None]
    key = torch.arange(n, device=q.device)[None, :]
    seen = (key <= pos) & ((key > pos - window) if window else (key >= 0))
    p = torch.softmax(x.masked_fill(~seen, -math.inf), dim=-1)
    o = torch.matmul(p.reshape(hkv, hq // hkv * t, n), v.contiguous()).reshape(hq, t, d)
    return o.transpose(0, 1).contiguous(), x, p


def _rotary(x, first, theta):
    t, _, d = x.shape
    freq = theta ** (-2.0 * torch.arange(d // 2, device=x.device, dtype=torch.float64) / d)
    angle = torch.arange(first, first + t, device=x.device, dtype=torch.float64)[:, None, None] * freq
    a, b = x[..., :d // 2], x[..., d // 2:]
    return torch.cat([a * angle.cos() - b * angle.sin(), b * angle.cos() + a * angle.sin()], dim=-1)


def _norm(x, w):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + float(torch.tensor(1e-6))) * w


def exact(case, seed):
    s = _inputs(case, seed)
    op, dbl = case["op"], torch.float64
    if op == "project":
        logits = torch.matmul(s["x"].to(dbl), s["w"].to(dbl).t())
        return {"tokens": logits.argmax(-1).to(torch.int32), "logits": logits}
    if op == "softcap":
        return {"logits": case["cap"] * torch.tanh(s["x"].to(dbl) / case["cap"])}
    hq, hkv, d, dt = case["hq"], case["hkv"], case["d"], _DT[case["dtype"]]
    scale, t = 1.0 / math.sqrt(d), case.get("tokens", 1)
    if op in ("append", "produce"):
        off = case["offset"]
        q, k, v = s["qp"].to(dbl), s["kp"].to(dbl), s["vp"]
        if op == "produce":
            q = _rotary(_norm(q, s["wq"].to(dbl)), off, 1e6)
            k = _rotary(_norm(k, s["wk"].to(dbl)), off, 1e6)
        q = q.to(dt)
        s["kc"][:, off:], s["vc"][:, off:] = k.to(dt).transpose(0, 1), v.to(dt).transpose(0, 1)
        o = _attend(q.to(dbl), s["kc"].to(dbl), s["vc"].to(dbl), off, scale)[0]
        r = {"context": o.reshape(-1), "k": s["kc"].to(dbl), "v": s["vc"].to(dbl)}
        return dict(r, q=q.to(dbl)) if op == "produce" else r
    if op == "attention":
        o, x, p = _attend(s["q"].to(dbl), s["k"].to(dbl).transpose(0, 1), s["v"].to(dbl).transpose(0, 1), 0, scale)
        keep = case["diag"]
        return {"context": o.reshape(-1), "scores": x.reshape(-1) if keep else None, "probs": p.reshape(-1) if keep else None}
    if op in ("decode_batch", "prefill_batch"):
        got = []
        for i, (o, n) in enumerate(zip(s["offsets"], s["lengths"])):
            k, v = (s[x][o:o + hkv * n * d].view(hkv, n, d).to(dbl) for x in ("k", "v"))
            got.append(_attend(s["q"][i].to(dbl), k, v, n - t, scale)[0].reshape(-1))
        return {"context": torch.cat(got)}
    if op == "ring":
        o = _attend(s["q"].to(dbl), s["k"].to(dbl), s["v"].to(dbl), case["committed"], scale, case["window"],
                    case["softcap"])[0]
        return {"context": o.reshape(-1)}
    if op == "window":
        o = _attend(s["q"].to(dbl), s["k"].to(dbl), s["v"].to(dbl), case["keys"] - t, scale, case["window"],
                    case["softcap"])[0]
        return {"context": o.reshape(-1)}
    got = {}
    for i, (q, k, v) in enumerate(s["layers"]):
        q, k = (_rotary(x.to(dbl), 0, 1e6).to(dt).to(dbl) for x in (q, k))
        o = _attend(q, k.transpose(0, 1), v.to(dt).to(dbl).transpose(0, 1), 0, scale, case["window"] if i < 5 else 0,
                    case["softcap"])[0]
        got["layer%d" % i] = o.reshape(o.shape[0], hq * d)
    return got
