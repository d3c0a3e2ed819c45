"""The work a user of this framework has it do, as cases that can be timed and checked.

A case is one pass of one layer's compressed-KV path through a public entry point:

  decode  a serving engine's decode step (Ops.append_decode): one new token per sequence is written to
          the paged cache and attention runs over it and everything before it
  write   the quantize-and-pack of a prefill chunk (Ops.write)
  extend  a serving engine's prefill step over cached history: attention of a ragged batch of new tokens
          (ExtendPlan.attend), then their write (ExtendPlan.write)
  chunk   a long prompt's chunk over its cached history (KushCache.attend_chunk)
  attend  one decode attention of a KushCache (KushCache.attend)
  prompt  causal attention of a first prompt over itself (hf.prompt_attention)

Keys are N(0, 1) plus a bias N(0, 6^2) on about a tenth of the channels of each kv head, values and queries
N(0, 1); a pool's blocks are handed out in random order, as in a server that has run for a while. Batches
are ragged around the case's length ("spread": a sequence has between (1 - spread) and 1 times it),
their lengths drawn from the case's "mix". The cached history is written by Ops.write itself.
"""
import math
import random

import torch

PAGE = 32
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ROWS = 1 << 17                               # history rows generated and written at a time


def listed():
    return [
        # a single user's chat, a few hundred tokens in: launch and latency
        dict(name="decode_one", kind="decode", batch=1, tokens=333, spread=0.0, mix=1, hkv=8, group=4, dim=128,
             bits=4, dtype="bf16", rot=True),
        # the headline decode: batch 64 at 4,096 tokens, 28 q heads over 4 kv heads
        dict(name="decode_batch", kind="decode", batch=64, tokens=4096, spread=0.0, mix=2, hkv=4, group=7, dim=128,
             bits=4, dtype="bf16", rot=False),
        # a busy server's step: 128 sequences of 256 to 8,192 tokens, int8 records
        dict(name="decode_ragged", kind="decode", batch=128, tokens=8192, spread=0.97, mix=3, hkv=8, group=4, dim=128,
             bits=8, dtype="bf16", rot=False),
        # long documents: 8 sequences of 131,072 tokens
        dict(name="decode_long", kind="decode", batch=8, tokens=131072, spread=0.0, mix=4, hkv=8, group=4, dim=128,
             bits=4, dtype="bf16", rot=True),
        # wide heads, many query heads per kv head, fp16 (one page stream of the matrix cores)
        dict(name="decode_wide", kind="decode", batch=19, tokens=6001, spread=0.5, mix=5, hkv=2, group=16, dim=256,
             bits=4, dtype="fp16", rot=True),
        # narrow heads, no head sharing to speak of, int8
        dict(name="decode_narrow", kind="decode", batch=33, tokens=2500, spread=0.9, mix=6, hkv=12, group=2, dim=64,
             bits=8, dtype="fp16", rot=False),
        # the chunked-prefill write of 8 prompts of 2,048 tokens, rotated (the int4 serving default)
        dict(name="write_prompts", kind="write", batch=8, tokens=2048, spread=0.0, history=0, mix=7, hkv=8, group=4,
             dim=128, bits=4, dtype="bf16", rot=True),
        # a mixed step's write: odd chunks, some onto a started page
        dict(name="write_ragged", kind="write", batch=13, tokens=611, spread=0.95, history=1000, mix=8, hkv=4, group=7,
             dim=128, bits=8, dtype="fp16", rot=False),
        # a serving prefill step: follow-up turns of 9 conversations over their cached history
        dict(name="extend_turns", kind="extend", batch=9, tokens=400, spread=0.9, history=8000, mix=9, hkv=8, group=4,
             dim=128, bits=4, dtype="bf16", rot=True),
        # a long prompt's chunk: 2,048 tokens over 32,768 cached ones
        dict(name="chunk_long", kind="chunk", batch=1, tokens=2048, history=32768 + 11, mix=10, hkv=8, group=4,
             dim=128, bits=4, dtype="bf16", rot=True),
        # the Hugging Face cache's decode attention, its default rotation, a small batch
        dict(name="attend_cache", kind="attend", batch=4, tokens=1000, mix=11, hkv=8, group=4, dim=128, bits=4,
             dtype="fp16", rot=True),
        # the first prompt of a batch
        dict(name="prompt_first", kind="prompt", batch=2, tokens=3001, mix=12, hkv=4, group=7, dim=128, bits=4,
             dtype="bf16", rot=True),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["decode"] * 4 + ["write", "write", "extend", "extend", "chunk", "attend", "prompt"])
    dim = rng.choice([64, 128, 128, 128, 256])
    c = dict(kind=kind, hkv=rng.choice([1, 2, 4, 8, 8, 12]), dim=dim, bits=rng.choice([4, 4, 8]),
             group=rng.choice([1, 2, 4, 4, 7, 8, 12, 16]), dtype=rng.choice(["bf16", "bf16", "bf16", "fp16", "fp16", "fp32"]),
             rot=rng.random() < 0.6, mix=rng.randrange(1 << 20))
    if kind == "decode":
        c["batch"] = _log(rng, 1, 200)
        # the tokens of a batch together: at most a third of the largest listed case's
        c["tokens"] = _log(rng, 20, max(40, min(131072, (1 << 20) // 3 * 8 // c["hkv"] * 128 // dim // c["batch"])))
        c["spread"] = rng.choice([0.0, 0.5, 0.95])
    elif kind == "write":
        c["batch"], c["tokens"] = _log(rng, 1, 40), _log(rng, 2, 4096)
        c["tokens"] = max(2, min(c["tokens"], 16384 * 8 // c["hkv"] * 128 // dim // c["batch"]))
        c["spread"], c["history"] = rng.choice([0.0, 0.9]), rng.choice([0, 0, _log(rng, 5, 4000)])
    elif kind == "extend":
        c["batch"], c["tokens"], c["history"] = _log(rng, 1, 16), _log(rng, 2, 1500), _log(rng, 1, 12000)
        c["spread"] = rng.choice([0.0, 0.9])
    elif kind == "chunk":
        c["batch"], c["tokens"] = rng.choice([1, 1, 2, 4]), _log(rng, 16, 2048)
        c["history"] = _log(rng, 30, 32768 // c["batch"])
    elif kind == "attend":
        c["batch"], c["tokens"] = _log(rng, 1, 32), _log(rng, 10, 8000)
    else:
        c["batch"], c["tokens"] = rng.choice([1, 1, 2, 4]), _log(rng, 20, 4096)
    if kind in ("extend", "chunk", "prompt"):
        # prefill runs in the model's half precision; its attention work at most the longest chunk's
        c["dtype"] = rng.choice(["bf16", "bf16", "fp16"])
        c["hkv"] = min(c["hkv"], max(1, 32 // c["group"]))
        while work(c)["flops"] > 1.1e12:
            c["tokens"] = max(2, c["tokens"] // 2)
    return c


# ------------------------------------------------------------------ sizes of a case
def _lengths(c):
    """(history, new) tokens of each sequence. A written chunk either starts on a page of its own or ends
    on a full one, so that a step can be repeated on the same cache."""
    rng = random.Random(c["mix"])
    spread = c.get("spread", 0.0)
    hist, new = [], []
    for _ in range(c["batch"]):
        n = max(1, round(c["tokens"] * (1 - spread * rng.random())))
        if c["kind"] == "decode":
            h, n = n - 1, 1
        elif c["kind"] in ("write", "extend"):
            h = round(c["history"] * (1 - spread * rng.random())) if c["history"] else 0
            if rng.random() < 0.5 or h < PAGE:
                h -= h % PAGE
            else:
                n = max(PAGE - h % PAGE, n - (h + n) % PAGE)
        else:
            h = c.get("history", 0)
        hist.append(h)
        new.append(n)
    return hist, new


def _record(c):
    row = c["dim"] if c["bits"] == 8 else c["dim"] // 2
    return 2 * PAGE * row + 4 * c["dim"] + 4 * PAGE


def work(c):
    """What one pass cannot do without: records and rows read once, results written once, and the
    products of q K^T and P V."""
    hist, new = _lengths(c)
    H, G, D, e, R = c["hkv"], c["group"], c["dim"], DTYPES[c["dtype"]].itemsize, _record(c)
    kind, bytes_, flops = c["kind"], 0, 0
    for h, n in zip(hist, new):
        total = h + n
        if kind in ("decode", "attend"):
            past = total - (total % PAGE if kind == "attend" else 0)
            bytes_ += H * (past // PAGE * R + (total % PAGE) * (R // (2 * PAGE) + D * e)) + 2 * H * G * D * e
            bytes_ += 2 * H * D * e * (kind == "decode")
            flops += 4 * H * G * D * total
            continue
        pairs = n * h + n * (n + 1) // 2
        if kind != "write":
            bytes_ += H * (h // PAGE * R + (h % PAGE) * (R // (2 * PAGE) + D * e)) + 2 * n * H * G * D * e
            flops += 4 * H * G * D * pairs
        bytes_ += 2 * n * H * D * e                                   # the new rows
        if kind in ("write", "extend"):
            done = total // PAGE - h // PAGE                           # K pages completed
            bytes_ += H * (done * (PAGE * (R - 4 * D - 4 * PAGE) // (2 * PAGE) + 4 * D)
                           + n * ((R - 4 * D - 4 * PAGE) // (2 * PAGE) + 4))
            bytes_ += H * D * e * ((h % PAGE) * (done > 0) + (total % PAGE) * (total // PAGE * PAGE >= h))
            flops += 10 * n * H * D
    return {"bytes": int(bytes_), "flops": int(flops)}


# ------------------------------------------------------------------ inputs
def _generator(seed, stream):
    g = torch.Generator(device="cuda")
    g.manual_seed((seed * 1000003 + stream * 7919 + 17) % (1 << 62))
    return g


def _biases(c, seed):
    g = _generator(seed, 1)
    H, D = c["hkv"], c["dim"]
    hit = torch.rand(H, D, generator=g, device="cuda") < 0.1
    return torch.where(hit, 6.0 * torch.randn(H, D, generator=g, device="cuda"), torch.zeros((), device="cuda"))


def _rows(c, seed, stream, n, bias):
    """n key rows and value rows [n, hkv, dim] of one sequence (or of one step's new tokens)."""
    g, dt, shape = _generator(seed, stream), DTYPES[c["dtype"]], (n, c["hkv"], c["dim"])
    k = (torch.randn(shape, generator=g, device="cuda") + bias).to(dt)
    return k, torch.randn(shape, generator=g, device="cuda").to(dt)


def _history(c, seed, s, n, bias):
    """The history of sequence s in pieces of at most ROWS rows: (first position, k, v)."""
    for i, at in enumerate(range(0, n, ROWS)):
        yield (at, *_rows(c, seed, 100 + 1000 * s + i, min(ROWS, n - at), bias))


def _new(c, seed, bias):
    """The step's new rows of all sequences, end to end, and its queries [rows, hkv * group, dim]."""
    total = sum(_lengths(c)[1])
    k, v = _rows(c, seed, 2, total, bias)
    q = torch.randn(total, c["hkv"] * c["group"], c["dim"], generator=_generator(seed, 3), device="cuda")
    return k, v, q.to(DTYPES[c["dtype"]])


def _ints(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


def _write_history(ops, c, seed, bias, hist, cache, block_table, tail_idx, tail_k):
    for s, h in enumerate(hist):
        for at, k, v in _history(c, seed, s, h, bias):
            n = k.shape[0]
            pages = torch.arange(at // PAGE, (at + n - 1) // PAGE + 1, dtype=torch.int32, device="cuda")
            ops.write(k, v, _ints([0, n]), _ints([at + n]), tail_idx[s:s + 1], torch.zeros_like(pages), pages,
                      cache, block_table[s:s + 1], tail_k, fused=True, rot=c["rot"])


def prepare(case, seed):
    """What a program holds before the call: the pool with the history in it, the step's rows and its plan."""
    from kushkash_amd import KushCache
    c, kind = case, case["kind"]
    dev, dt = torch.device("cuda"), DTYPES[c["dtype"]]
    H, G, D = c["hkv"], c["group"], c["dim"]
    hist, new = _lengths(c)
    bias = _biases(c, seed)
    scale = 1.0 / math.sqrt(D)
    if kind in ("chunk", "attend", "prompt"):
        B, T = c["batch"], c["tokens"]
        k, v, q = (x.view(B, T, -1, D) for x in _new(c, seed, bias))
        st = dict(case=c, scale=scale)
        if kind != "attend":
            st.update((n, x.transpose(1, 2)) for n, x in (("q", q), ("k", k), ("v", v)))
        else:
            st["q"] = q[:, -1].contiguous()
        if kind != "prompt":
            n = c["history"] if kind == "chunk" else T
            st["cache"] = KushCache(1, H, H * G, D, batch_size=B, bits=c["bits"], device=dev, dtype=dt,
                                    max_length=n, rotate=c["rot"])
            if kind == "attend":
                st["cache"].write(0, k.transpose(1, 2), v.transpose(1, 2))
            else:
                for at in range(0, n, ROWS):
                    ks, vs = zip(*(list(_history(c, seed, b, n, bias))[at // ROWS][1:] for b in range(B)))
                    st["cache"].write(0, torch.stack(ks).transpose(1, 2), torch.stack(vs).transpose(1, 2))
        return st

    from kushkash_amd import Ops, record_bytes
    ops = Ops(dev, D, c["bits"], G, dt)
    S = c["batch"]
    pages = [-(-(h + n) // PAGE) for h, n in zip(hist, new)]
    blocks = torch.randperm(sum(pages) + 7, generator=_generator(seed, 4), device="cuda").to(torch.int32)
    block_table = torch.zeros(S, max(pages), dtype=torch.int32, device=dev)
    at = 0
    for s, p in enumerate(pages):
        block_table[s, :p] = blocks[at:at + p]
        at += p
    cache = torch.zeros(blocks.numel(), H, record_bytes(D, c["bits"]), dtype=torch.uint8, device=dev)
    tail_k = torch.zeros(S, H, PAGE, D, dtype=dt, device=dev)
    tail_idx = torch.arange(S, dtype=torch.int32, device=dev)
    _write_history(ops, c, seed, bias, hist, cache, block_table, tail_idx, tail_k)
    k, v, q = _new(c, seed, bias)
    st = dict(case=c, scale=scale, ops=ops, k=k, v=v, q=q, cache=cache, block_table=block_table, tail_k=tail_k,
              tail_idx=tail_idx, seq_lens=_ints([h + n for h, n in zip(hist, new)]))
    if kind == "decode":
        st["out"] = torch.empty_like(q)
        st["splits"] = ops.splits(S, H, max(pages))
        st["work"] = torch.empty(S * H * st["splits"] * G * (D + 2), dtype=torch.float32, device=dev)
        longest = sorted(range(S), key=lambda s: -(hist[s] + new[s]))
        st["order"] = _ints(longest) if len(set(pages)) > 1 else None
    else:
        from kushkash_amd._prefill import ExtendPlan
        st["plan"] = ExtendPlan.build(new, hist, list(range(S)), block_table, kv_heads=H, head_dim=D, dtype=dt)
    return st


def run(st):
    c = st["case"]
    kind = c["kind"]
    if kind == "chunk":
        return {"out": st["cache"].attend_chunk(0, st["q"], st["k"], st["v"])}
    if kind == "attend":
        return {"out": st["cache"].attend(0, st["q"])}
    if kind == "prompt":
        from kushkash_amd.hf import prompt_attention
        return {"out": prompt_attention(st["q"], st["k"], st["v"], st["scale"])}
    ops, cache, bt, tail = st["ops"], st["cache"], st["block_table"], st["tail_k"]
    if kind == "decode":
        ops.append_decode(st["k"], st["v"], st["q"], st["out"], cache, bt, st["seq_lens"], st["tail_idx"], tail,
                          st["scale"], st["splits"], st["work"], order=st["order"], rot=c["rot"])
        return {"out": st["out"], "cache": cache, "tail_k": tail}
    plan = st["plan"]
    out = {}
    if kind == "extend":
        out["out"] = plan.attend(ops, st["q"], st["k"], st["v"], cache, tail, bt, st["tail_idx"], st["scale"],
                                 c["rot"])
    plan.write(ops, st["k"], st["v"], st["seq_lens"], st["tail_idx"], cache, bt, tail, c["rot"])
    return {**out, "cache": cache, "tail_k": tail}


# ------------------------------------------------------------------ what outputs may differ by
def tolerance(c):
    """A write's records are whole numbers and its K tails copies: exact. Attention: four times what the
    path was measured to be from 64-bit arithmetic on the same inputs, which is the output's rounding
    and, where the cache rotates or the history is unpacked, the one of q, k, v rows to the model's type."""
    if c["kind"] == "write":
        return "exact"
    rel = {"bf16": 8e-3, "fp16": 1.2e-3, "fp32": 5.5e-4}[c["dtype"]]
    if c["kind"] in ("extend", "chunk"):
        rel = {"bf16": 1.6e-2, "fp16": 2.5e-3}[c["dtype"]]
    elif c["rot"]:
        rel *= 1.5
    return {"rel": rel}


# ------------------------------------------------------------------ the same in plain torch, in 64 bits
def _wht(x):
    """Walsh-Hadamard transform of the last dim, strides 1, 2, 4, ..., then 1 / sqrt(D), in x's type."""
    D, y, stride = x.shape[-1], x, 1
    while stride < D:
        y = y.view(*x.shape[:-1], D // (2 * stride), 2, stride)
        y = torch.stack((y[..., 0, :] + y[..., 1, :], y[..., 0, :] - y[..., 1, :]), -2).reshape(x.shape)
        stride *= 2
    return y * torch.tensor(1.0 / math.sqrt(D), dtype=x.dtype)


def _quantized(x, dim, bits):
    """x [..., 32 or more rows grouped, ...] quantized over `dim` by the record format's fp32 arithmetic
    (fp16 scale and bias), as its values in 64 bits."""
    half, levels = 1 << (bits - 1), (1 << bits) - 1
    mn, mx = x.amin(dim, keepdim=True), x.amax(dim, keepdim=True)
    s = ((mx - mn) / torch.full_like(mn, levels)).half().float()
    b = (mn + s * half).half().float()
    inv = torch.where(s > 0, 1.0 / s, torch.zeros_like(s))
    return torch.round((x - b) * inv).clamp(-half, half - 1).double() * s.double() + b.double()


def _cached(c, k, v):
    """The cached keys and values of rows k, v [n, hkv, dim] (all of one sequence), in 64 bits and
    unrotated: whole pages of K per channel, the rest exact, V per token."""
    n, dt = k.shape[0], k.dtype
    full = n // PAGE * PAGE
    k, v = ((_wht(x.float()).to(dt) if c["rot"] else x).float() for x in (k, v))
    kq = _quantized(k[:full].view(-1, PAGE, *k.shape[1:]), 1, c["bits"]).view(full, *k.shape[1:])
    kd, vd = torch.cat([kq, k[full:].double()]), _quantized(v, 2, c["bits"])
    return (_wht(kd), _wht(vd)) if c["rot"] else (kd, vd)


def _attention(q, k, v, scale):
    """Causal attention of the last T of N positions: q [T, heads, dim], k, v [N, hkv, dim], 64 bits."""
    T, N, G = q.shape[0], k.shape[0], q.shape[1] // k.shape[1]
    out = torch.empty_like(q)
    step = max(1, (1 << 28) // N)
    for h in range(q.shape[1]):
        kh, vh = k[:, h // G].t().contiguous(), v[:, h // G].contiguous()
        for t in range(0, T, step):
            x = torch.mm(q[t:t + step, h], kh).mul_(scale)
            if T > 1:
                rows = torch.arange(t, t + x.shape[0], device=x.device)[:, None] + (N - T)
                x.masked_fill_(torch.arange(N, device=x.device)[None, :] > rows, -math.inf)
            out[t:t + step, h] = torch.mm(torch.softmax(x, -1), vh)
    return out


def exact(case, seed):
    c, kind = case, case["kind"]
    if kind == "write":
        return None
    hist, new = _lengths(c)
    bias = _biases(c, seed)
    k, v, q = _new(c, seed, bias)
    scale = 1.0 / math.sqrt(c["dim"])
    outs, at = [], 0
    for s, (h, n) in enumerate(zip(hist, new)):
        if kind == "decode" or kind == "attend":                        # the new rows are in the cache
            rows = [r[1:] for r in _history(c, seed, s, h, bias)] + [(k[at:at + n], v[at:at + n])]
            kk, vv = _cached(c, torch.cat([r[0] for r in rows]), torch.cat([r[1] for r in rows]))
        else:
            kk, vv = k[at:at + n].double(), v[at:at + n].double()
            if h:
                rows = [r[1:] for r in _history(c, seed, s, h, bias)]
                hk, hv = _cached(c, torch.cat([r[0] for r in rows]), torch.cat([r[1] for r in rows]))
                kk, vv = torch.cat([hk, kk]), torch.cat([hv, vv])
        qs = q[at + n - 1:at + n] if kind == "attend" else q[at:at + n]
        outs.append(_attention(qs.double(), kk, vv, scale))
        at += n
    if kind in ("decode", "extend"):
        return {"out": torch.cat(outs), "cache": None, "tail_k": None}
    if kind == "attend":
        return {"out": torch.cat(outs)}
    return {"out": torch.stack(outs).transpose(1, 2)}
