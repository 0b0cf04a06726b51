"""What is measured: attention calls as a serving or training program makes them.

Each case is one call of the public v2 / v3 API (forward, or forward and
backward) on inputs that such a program holds on the GPU. The fields of a case:

  path    "kvcache" (decode, speculative verification and chunked prefill
          against a cache), "dense" or "varlen"
  api     2 or 3: the flash_attn_npu_v2 or flash_attn_npu_v3 package
  train   forward and backward; the gradients of q, k and v are results
  dtype   "bf16", "fp16" or "fp8" (e4m3 inputs with descales, bf16 results)
  B, Sq, H, Hk, D   sequences, query positions (the longest for varlen),
          query heads, key / value heads, head dimension
  Sk      dense: keys; kvcache: rows of a contiguous cache (0: paged)
  lo, hi  lengths in the cache (kvcache) or of the sequences (varlen), drawn
          from [lo, hi] over their logarithm by `lens`, a seed of its own, so
          that the work of a case does not depend on the seed of its values
  page    rows per block of a paged cache, 0 for a contiguous one
  new     tokens that the call appends to the cache
  rotary  NeoX rotary embedding over the whole head dimension
  causal, left (left window, -1: none), softcap (0: none), alibi
"""
import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash-attention-npu_amd"))

import flash_attn_npu_v2 as v2  # noqa: E402
import flash_attn_npu_v3 as v3  # noqa: E402

DEVICE = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp8": torch.float8_e4m3fn}
DEFAULTS = dict(path="dense", api=2, train=False, dtype="bf16", B=1, Sq=1, H=32, Hk=8, D=128, Sk=0, lo=0, hi=0, lens=0,
                page=0, new=0, rotary=False, causal=True, left=-1, softcap=0.0, alibi=False)
# no drawn case costs more than the largest listed ones (train_dense, decode_paged)
MOST_FLOPS, MOST_BYTES = 1.9e12, 2.5e9


def _case(**kw):
    return dict(DEFAULTS, **kw)


def listed():
    return [
        # one user's next token: a short cache, nothing to fill the chip with
        _case(name="decode_one", path="kvcache", B=1, Sk=2048, lo=777, hi=777, new=1),
        # a serving step of 32 users with contiguous caches
        _case(name="decode_batch", path="kvcache", B=32, Sk=8192, lo=1024, hi=8191, lens=2, new=1),
        # a serving step over a paged cache with lengths of every size
        _case(name="decode_paged", path="kvcache", api=3, B=64, H=64, page=256, lo=512, hi=32768, lens=3, new=1),
        # the same with an e4m3 cache
        _case(name="decode_paged_fp8", path="kvcache", api=3, dtype="fp8", B=64, H=64, page=256, lo=512, hi=32768,
              lens=3, new=1),
        # verification of 4 speculated tokens, sliding window and ALiBi over long contexts
        _case(name="verify_window", path="kvcache", B=8, Sq=4, page=256, lo=16384, hi=65536, lens=5, left=4096,
              alibi=True),
        # a prompt's next chunk with rotary, appended behind what the cache holds
        _case(name="chunked_prefill", path="kvcache", B=4, Sq=2048, Sk=8192, lo=6144, hi=6144, new=2048, rotary=True),
        # a short prompt, little work for each compute unit
        _case(name="dense_small", dtype="fp16", B=2, Sq=512, Sk=512, H=16, Hk=16),
        # an fp8 prompt
        _case(name="dense_fp8", api=3, dtype="fp8", B=2, Sq=4096, Sk=4096),
        # a training step of a causal grouped-query layer
        _case(name="train_dense", train=True, B=4, Sq=4096, Sk=4096),
        # a training step over packed documents of uneven length
        _case(name="train_varlen", path="varlen", api=3, train=True, B=24, Sq=2048, H=16, lo=64, hi=2048, lens=8),
        # a training step of a bidirectional encoder, odd length, head dimension 64
        _case(name="train_encoder", train=True, dtype="fp16", B=8, Sq=1025, Sk=1025, H=16, Hk=16, D=64, causal=False),
        # a training step with head dimension 256, sliding window and soft cap
        _case(name="train_d256", train=True, B=2, Sq=4096, Sk=4096, H=16, D=256, left=1024, softcap=30.0),
    ]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def _draw(rng):
    kind = rng.choice(["decode", "decode", "verify", "chunked", "dense", "train_dense", "train_dense", "train_varlen"])
    lens = rng.randrange(1 << 20)
    if kind in ("decode", "verify"):
        hk = rng.choice([2, 4, 8, 8, 16])
        lo, hi = sorted((_log(rng, 128, 32768), _log(rng, 128, 32768)))
        page = rng.choice([0, 64, 128, 256])
        c = _case(path="kvcache", api=rng.choice([2, 3]), dtype=rng.choice(["bf16", "bf16", "fp16", "fp8"]),
                  B=_log(rng, 1, 64), H=hk * rng.choice([1, 4, 4, 8]), Hk=hk, D=rng.choice([64, 128, 128]), lo=lo, hi=hi,
                  lens=lens, page=page, Sk=0 if page else hi + 8, new=1)
        if kind == "verify":
            c.update(Sq=rng.choice([2, 3, 4]), H=hk * 4, new=0, left=rng.choice([-1, 1024, 4096]),
                     lo=max(c["lo"], 8), alibi=c["api"] == 2 and rng.random() < 0.5)
        if c["dtype"] == "fp8":
            c.update(api=3, alibi=False)
        return c
    if kind == "chunked":
        sq, past = _log(rng, 64, 2048), _log(rng, 16, 6144)
        page = rng.choice([0, 64, 256])
        return _case(path="kvcache", api=rng.choice([2, 3]), B=_log(rng, 1, 8), Sq=sq, lo=past, hi=past, lens=lens,
                     page=page, Sk=0 if page else past + sq, new=sq, rotary=rng.random() < 0.7)
    d = rng.choice([64, 96, 128, 128, 256])
    hk = rng.choice([4, 8, 16])
    c = _case(api=rng.choice([2, 3]), train=kind != "dense", dtype=rng.choice(["bf16", "bf16", "fp16"]),
              H=hk * rng.choice([1, 2, 4]), Hk=hk, D=d, causal=rng.random() < 0.75)
    if kind == "train_varlen":
        lo, hi = sorted((_log(rng, 32, 4096), _log(rng, 32, 4096)))
        c.update(path="varlen", B=_log(rng, 2, 32), lo=lo, hi=hi, Sq=hi, lens=lens)
    else:
        s = _log(rng, 64, 4096)
        c.update(B=_log(rng, 1, 8), Sq=s, Sk=s)
        if not c["train"] and rng.random() < 0.3:
            c.update(dtype="fp8", api=3)
        if c["causal"] and rng.random() < 0.25:
            c["left"] = rng.choice([256, 1024])
        if rng.random() < 0.2:
            c["softcap"] = rng.choice([15.0, 30.0, 50.0])
    return c


def draw(rng):
    while True:
        c = _draw(rng)
        w = work(c)
        if w["flops"] <= MOST_FLOPS and w["bytes"] <= MOST_BYTES:
            return c


def _lengths(c):
    r = random.Random(c["lens"])
    return [_log(r, c["lo"], c["hi"]) if c["hi"] > c["lo"] else c["lo"] for _ in range(c["B"])]


def _shapes(c):
    """(query positions, keys) of each sequence."""
    if c["path"] == "dense":
        return [(c["Sq"], c["Sk"])] * c["B"]
    if c["path"] == "varlen":
        return [(n, n) for n in _lengths(c)]
    return [(c["Sq"], n + c["new"]) for n in _lengths(c)]


def _seen(c, sq, sk):
    """(pairs that the mask leaves, keys that some query sees)."""
    i = torch.arange(sq, dtype=torch.int64) + (sk - sq)
    hi = i.clamp(max=sk - 1) if c["causal"] else torch.full_like(i, sk - 1)
    lo = (i - c["left"]).clamp(min=0) if c["left"] >= 0 else torch.zeros_like(i)
    return int((hi - lo + 1).clamp(min=0).sum()), int(hi.max() - lo.min() + 1)


def work(c):
    es = 1 if c["dtype"] == "fp8" else 2
    pairs = rows = keys = 0
    known = {}
    for s in _shapes(c):
        p, k = known.setdefault(s, _seen(c, *s))
        pairs, rows, keys = pairs + p, rows + s[0], keys + k
    q, kv = rows * c["H"] * c["D"], keys * c["Hk"] * c["D"]
    moved = q * es + 2 * kv * es + q * 2 + rows * c["H"] * 4          # q, k, v; out, lse
    if c["new"]:
        moved += 2 * c["B"] * c["new"] * c["Hk"] * c["D"] * es        # appended rows, written once
    if c["train"]:
        moved += 2 * q * es + 2 * kv * es                             # dout, dq, dk, dv
    return {"bytes": moved, "flops": pairs * c["H"] * c["D"] * (14 if c["train"] else 4)}


def tolerance(c):
    # 16-bit results of the same sums in another order: a unit in the last
    # place on part of the values, and P and dS rounded at other maxima (about
    # 3e-4 from 64 bits in fp16, 2.5e-3 in bf16)
    return {"rel": 1.2e-3, "max": 0.05} if c["dtype"] == "fp16" else {"rel": 1e-2, "max": 0.2}


def _random(g, dtype, *shape):
    if dtype != torch.float8_e4m3fn:
        return torch.empty(shape, dtype=dtype, device=DEVICE).normal_(generator=g)
    return torch.empty(shape, dtype=torch.bfloat16, device=DEVICE).normal_(generator=g).to(dtype)


def prepare(c, seed):
    g = torch.Generator(device=DEVICE)
    g.manual_seed(seed)
    dt, B, H, Hk, D = DTYPES[c["dtype"]], c["B"], c["H"], c["Hk"], c["D"]
    fp8, s = c["dtype"] == "fp8", {}
    i32 = dict(dtype=torch.int32, device=DEVICE)
    if c["path"] == "varlen":
        n = _lengths(c)
        s["cu"] = torch.tensor([sum(n[:i]) for i in range(B + 1)], **i32)
        s["max"] = max(n)
        q, kv = (sum(n), H, D), (sum(n), Hk, D)
    elif c["path"] == "dense":
        q, kv = (B, c["Sq"], H, D), (B, c["Sk"], Hk, D)
    else:
        n = _lengths(c)
        s["lens"] = torch.tensor(n, **i32)
        q, kv = (B, c["Sq"], H, D), (B, c["Sk"], Hk, D)
        if c["page"]:
            need = [-(-(x + c["new"]) // c["page"]) for x in n]
            blocks = torch.randperm(sum(need) + 4, generator=g, device=DEVICE).to(torch.int32).tolist()
            table = [[0] * max(need) for _ in n]
            for row, m in zip(table, need):
                row[:m] = [blocks.pop() for _ in range(m)]
            s["table"] = torch.tensor(table, **i32)
            kv = (sum(need) + 4, c["page"], Hk, D)
    s["q"], s["k"], s["v"] = _random(g, dt, *q), _random(g, dt, *kv), _random(g, dt, *kv)
    if c["new"]:
        s["k_new"], s["v_new"] = _random(g, dt, B, c["new"], Hk, D), _random(g, dt, B, c["new"], Hk, D)
    if c["rotary"]:
        rate = 10000.0 ** (-torch.arange(0, D, 2, dtype=torch.float64, device=DEVICE) / D)
        angle = torch.arange(c["hi"] + c["new"], dtype=torch.float64, device=DEVICE)[:, None] * rate
        s["cos"], s["sin"] = angle.cos().to(dt), angle.sin().to(dt)
    if c["alibi"]:
        s["slopes"] = torch.tensor([2.0 ** (-8.0 * (h + 1) / H) for h in range(H)], device=DEVICE)
    if fp8:
        for name in ("q_descale", "k_descale", "v_descale"):
            s[name] = torch.empty(B, Hk, device=DEVICE).uniform_(0.75, 1.25, generator=g)
    if c["train"]:
        s["dout"] = _random(g, dt, *q)
        for x in ("q", "k", "v"):
            s[x].requires_grad_(True)
    s["case"] = c
    return s


def run(s):
    c = s["case"]
    how = dict(causal=c["causal"], window_size=(c["left"], 0 if c["left"] >= 0 else -1), softcap=c["softcap"])
    if c["dtype"] == "fp8":
        how.update(q_descale=s["q_descale"], k_descale=s["k_descale"], v_descale=s["v_descale"])
    if c["path"] == "kvcache":
        more = dict(cache_seqlens=s["lens"], return_softmax_lse=True)
        if c["new"]:
            more.update(k=s["k_new"], v=s["v_new"])
        if c["rotary"]:
            more.update(rotary_cos=s["cos"], rotary_sin=s["sin"], rotary_interleaved=False)
        if c["api"] == 2:
            r = v2.flash_attn_with_kvcache(s["q"], s["k"], s["v"], block_table=s.get("table"),
                                           alibi_slopes=s.get("slopes"), **more, **how)
        else:
            r = v3.flash_attn_with_kvcache(s["q"], s["k"], s["v"], page_table=s.get("table"), **more, **how)
        return {"out": r[0], "lse": r[1], **({"k": s["k"], "v": s["v"]} if c["new"] else {})}
    api = v2 if c["api"] == 2 else v3
    if c["path"] == "varlen":
        out = api.flash_attn_varlen_func(s["q"], s["k"], s["v"], s["cu"], s["cu"], s["max"], s["max"], **how)
    else:
        out = api.flash_attn_func(s["q"], s["k"], s["v"], **how)
    if not c["train"]:
        return {"out": out}
    dq, dk, dv = torch.autograd.grad(out, (s["q"], s["k"], s["v"]), s["dout"])
    return {"out": out, "dq": dq, "dk": dk, "dv": dv}


def _rotate(x, cos, sin):
    a, b = x.chunk(2, dim=-1)
    return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)


def _attend(c, q, k, v, slope):
    """One sequence and key / value head in 64 bits: q (Sq, g, D), k and v (Sk, D); out and lse."""
    sq, sk = q.shape[0], k.shape[0]
    x = torch.matmul(q.reshape(-1, q.shape[-1]), k.t()).view(sq, -1, sk) * c["D"] ** -0.5
    if c["softcap"]:
        x = c["softcap"] * torch.tanh(x / c["softcap"])
    i = torch.arange(sk - sq, sk, device=q.device)[:, None]
    j = torch.arange(sk, device=q.device)[None]
    if slope is not None:
        x = x - slope[None, :, None] * (i - j).abs()[:, None]
    hidden = torch.zeros(sq, sk, dtype=torch.bool, device=q.device)
    if c["causal"] or c["left"] >= 0:
        hidden |= j > i
    if c["left"] >= 0:
        hidden |= j < i - c["left"]
    x = x.masked_fill(hidden[:, None], -math.inf)
    lse = torch.logsumexp(x, dim=-1)
    p = torch.exp(x - lse[..., None])
    return torch.matmul(p.view(-1, sk), v).view(sq, -1, v.shape[-1]), lse


def exact(c, seed):
    s = prepare(c, seed)
    H, Hk = c["H"], c["Hk"]
    g = H // Hk
    q = s["q"].detach().double()
    out = torch.zeros_like(q)
    shapes = _shapes(c)
    if c["path"] == "kvcache":
        k, v, n = s["k"].detach().clone(), s["v"].detach().clone(), _lengths(c)
        if c["rotary"]:  # rotated rows are kept in 64 bits
            k, v = k.double(), v.double()
        places = []
        for b, (_, sk) in enumerate(shapes):
            at = torch.arange(sk, device=DEVICE)
            places.append((s["table"][b].long()[at // c["page"]], at % c["page"]) if c["page"]
                          else (torch.full_like(at, b), at))
            if c["new"]:
                at = tuple(x[n[b]:] for x in places[b])
                kn = s["k_new"][b]
                if c["rotary"]:
                    cos, sin = (s[x].double()[n[b]:sk] for x in ("cos", "sin"))
                    kn = _rotate(kn.double(), cos[:, None], sin[:, None])
                    q[b] = _rotate(q[b], cos[:, None], sin[:, None])
                _bytes(k)[at], _bytes(v)[at] = _bytes(kn), _bytes(s["v_new"][b].to(v.dtype))
        lse = torch.zeros(c["B"], H, c["Sq"], dtype=torch.float64, device=DEVICE)
    else:
        k, v, lse = s["k"].detach().double(), s["v"].detach().double(), None
    if c["train"]:
        dq, dk, dv = torch.zeros_like(q), torch.zeros_like(k), torch.zeros_like(v)
    start = 0
    for b, (sq, sk) in enumerate(shapes):
        rows = slice(start, start + sq) if c["path"] == "varlen" else (b,)
        keys = places[b] if c["path"] == "kvcache" else rows
        start += sq
        first = max(0, sk - sq - c["left"]) if c["left"] >= 0 else 0  # keys before it are seen by no query
        if c["path"] == "kvcache":
            keys = tuple(x[first:] for x in keys)
            kb, vb = (_bytes(x)[keys].view(x.dtype).double() for x in (k, v))
            view = dict(c)
        else:
            kb, vb, view = k[keys], v[keys], c
        for h in range(Hk):
            heads = slice(h * g, (h + 1) * g)
            qh, kh, vh = q[rows][:, heads], kb[:, h], vb[:, h]
            if c["dtype"] == "fp8":
                qh, kh, vh = qh * s["q_descale"][b, h], kh * s["k_descale"][b, h], vh * s["v_descale"][b, h]
            slope = s["slopes"].double()[heads] if c["alibi"] else None
            if not c["train"]:
                o, l = _attend(view, qh, kh, vh, slope)
                out[rows][:, heads] = o
                if lse is not None:
                    lse[b, heads] = l.t()
                continue
            qh, kh, vh = (x.detach().requires_grad_(True) for x in (qh, kh, vh))
            o, _ = _attend(view, qh, kh, vh, slope)
            grads = torch.autograd.grad(o, (qh, kh, vh), s["dout"][rows][:, heads].double())
            out[rows][:, heads] = o.detach()
            dq[rows][:, heads], dk[keys][:, h], dv[keys][:, h] = grads
    if c["path"] == "kvcache":
        r = {"out": out, "lse": lse}
        return {**r, "k": k, "v": v} if c["new"] else r
    return {"out": out, "dq": dq, "dk": dk, "dv": dv} if c["train"] else {"out": out}


def _bytes(x):
    """e4m3 values as bytes, which can be indexed; others as they are."""
    return x.view(torch.uint8) if x.dtype == torch.float8_e4m3fn else x
