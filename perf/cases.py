"""The workloads the framework's speed is measured on: one layer's share of serving steps, each through
kvq.cuda_kernels as a serving program (the vLLM backend of this package) calls it.

A case is a dict of plain values; its request lengths follow from the case alone (`lens_seed`), its
tensors from the seed. Caches hold codes of the model-like distribution the benchmark uses (K with
log-normal channel gains, V and q normal), laid out as vLLM lays them out ([num_blocks, H, block, 2 D],
K and V interleaved) or as two separate [num_blocks, block, H, D] arrays; pages are shuffled.

Kinds:
  write   quantize a step's new K / V rows and scatter them into the paged cache
  short   INT8 attention of decode (1 query token) and verification (2..8 tokens) requests; split
          buffers are kept by the program and passed where the backend would pass them
  step    one attention call of a step with long-query requests (prefill, chunked prefill), alone or
          beside decode requests; the plan is made once per step, outside the layer's call
  graph   `layers` layers of a decode step (cache write + attention) captured in one HIP graph, replayed
"""
import math
import os
import random
import sys

import numpy as np
import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "int8-kvcache_amd"))
from kvq import cuda_kernels as ck  # noqa: E402

DEV = "cuda"
ABSMAX = 3.8        # calibration maximum of a channel, in standard deviations (4,096 normal samples)
CHUNK = 1 << 25     # elements drawn at a time
FAR = 1 << 17       # mixes a case's seeds apart


def _case(name, kind, **kw):
    c = dict(name=name, kind=kind, hq=28, hkv=4, d=128, block=16, vllm=True, per_channel=True,
             requests=0, query=1, lo=1, hi=1, lens_seed=1,      # short-query requests, keys log-uniform in [lo, hi]
             chunks="",                                         # long requests: "query:keys query:keys ..."
             tokens=0, pad=0.0, layers=1)
    c.update(kw)
    return c


def listed():
    return [
        # the cache write of a decode step: 32 requests' one new token each (launch latency)
        _case("write_step_32", "write", tokens=32),
        # the cache write of a prefill step, the benchmark's size: 16,384 tokens, 2% of the slots padding
        _case("write_prefill_16384", "write", tokens=16384, pad=0.02),
        # a ragged chunk of a small model with head_dim 64 and 2 kv heads, one scale per head
        _case("write_d64_3001", "write", hq=14, hkv=2, d=64, tokens=3001, pad=0.02, per_channel=False, vllm=False),
        # one user's decode at a moderate context: the smallest attention call
        _case("decode_1x4096", "short", requests=1, lo=4096, hi=4096),
        # the headline workload: 128 requests of 32k keys, bound by memory bandwidth
        _case("decode_128x32768", "short", requests=128, lo=32768, hi=32768),
        # a serving batch of very unequal contexts, 1 key to 32k
        _case("decode_96_ragged", "short", hq=32, hkv=8, requests=96, lo=1, hi=32768, lens_seed=9),
        # speculative decoding: 64 requests verify 8 tokens each (56 query rows per kv head)
        _case("verify_64x8", "short", requests=64, query=8, lo=512, hi=8192, lens_seed=7),
        # a short draft: 4 tokens each (28 query rows per kv head), larger blocks, separate caches
        _case("verify_24x4_block32", "short", requests=24, query=4, lo=300, hi=6000, lens_seed=5, block=32, vllm=False),
        # chunked prefill: the next 512 tokens of one request at 8k keys
        _case("chunk_512_of_8192", "step", chunks="512:8192"),
        # a mixed step: two prompts being read (one from its start, one mid-way) beside 48 decoding requests
        _case("mixed_48_decode_2_prompts", "step", hq=32, hkv=8, requests=48, lo=16, hi=8192, lens_seed=3,
              chunks="700:700 333:2500"),
        # four whole 16k prompts at once: bound by the matrix cores
        _case("prefill_4x16384", "step", hq=32, hkv=8, chunks="16384:16384 16384:16384 16384:16384 16384:16384"),
        # small-batch decode as it is served: captured, the layers back to back
        _case("graph_8x2k_4_layers", "graph", requests=8, lo=1000, hi=3000, lens_seed=2, layers=4),
    ]


HEADS = [(28, 4, 128), (32, 8, 128), (14, 2, 64), (12, 2, 128), (16, 16, 64)]


def _log(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    hq, hkv, d = rng.choice(HEADS)
    base = dict(hq=hq, hkv=hkv, d=d, block=rng.choice([16, 16, 32, 64]), vllm=rng.random() < 0.7,
                per_channel=rng.random() < 0.75, lens_seed=rng.randrange(1000))
    kind = rng.choice(["write", "short", "short", "step", "step", "graph"])
    if kind == "write":
        c = _case("", kind, tokens=_log(rng, 1, 16384), pad=rng.choice([0.0, 0.02, 0.3]), **base)
    elif kind == "short":
        query = rng.choice([1, 1, 1, 2, 3, 5, 8])
        requests = _log(rng, 1, 128)
        hi = max(64, min(32768, int(2 ** 21 / requests), int(2 ** 21 / (requests * hkv / 4))))
        lo = rng.choice([1, max(1, hi // 16), hi])
        c = _case("", kind, query=query, requests=requests, lo=max(lo, query), hi=max(hi, query), **base)
    elif kind == "step":
        chunks = []
        for _ in range(rng.choice([1, 1, 2, 3])):
            q = _log(rng, 9, 4096)
            chunks.append("%d:%d" % (q, q + rng.choice([0, _log(rng, 1, 16384)])))
        c = _case("", kind, requests=rng.choice([0, _log(rng, 1, 64)]), lo=1, hi=8192, chunks=" ".join(chunks), **base)
    else:
        c = _case("", kind, requests=_log(rng, 1, 32), lo=64, hi=4096, layers=rng.choice([2, 4]), **base)
    del c["name"]
    return c


# ------------------------------------------------------------------------------------------------ shapes
def _lens(c):
    """(query lengths, key counts) of the requests, short-query ones first (the backend orders them so)."""
    r = random.Random(c["lens_seed"])
    keys = [min(c["hi"], max(c["lo"], _log(r, c["lo"], c["hi"]))) for _ in range(c["requests"])]
    q = [c["query"]] * c["requests"]
    for part in c["chunks"].split():
        a, b = part.split(":")
        q.append(int(a))
        keys.append(int(b))
    return q, keys


def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed(int(seed) * FAR + what)


def _codes(shape, g):
    """int8 codes of a normal channel with scale ABSMAX / 127."""
    out = torch.empty(shape, dtype=torch.int8, device=DEV)
    flat = out.view(-1)
    for s in range(0, flat.numel(), CHUNK):
        n = min(CHUNK, flat.numel() - s)
        x = torch.randn(n, generator=g, device=DEV)
        flat[s:s + n] = x.mul_(127.0 / ABSMAX).round_().clamp_(-127, 127).to(torch.int8)
    return out


def _static(c, seed):
    g = _gen(seed, 1)
    hkv, d = c["hkv"], c["d"]
    gain = torch.exp(torch.randn(hkv, d, generator=g, device=DEV))
    mu = 0.5 * torch.randn(hkv, d, generator=g, device=DEV)
    ks = gain * (ABSMAX / 127) if c["per_channel"] else torch.full((hkv, 1), 2.0 * ABSMAX / 127, device=DEV)
    vs = (1 + 0.1 * torch.rand(hkv, d if c["per_channel"] else 1, generator=g, device=DEV)) * (ABSMAX / 127)
    return {"k_scale": ks.contiguous(), "v_scale": vs.contiguous(), "k_mu": mu.contiguous()}, gain


def _views(c, kv):
    """K and V as the operators take them, [num_blocks, block, H, D]."""
    if c["vllm"]:
        by_slot = kv.permute(0, 2, 1, 3)
        return by_slot[..., :c["d"]], by_slot[..., c["d"]:]
    return kv[0], kv[1]


def _cache_shape(c, blocks):
    return (blocks, c["hkv"], c["block"], 2 * c["d"]) if c["vllm"] else (2, blocks, c["block"], c["hkv"], c["d"])


def _table(c, keys, seed):
    """Block table [requests, pages] with shuffled pages, and the blocks of the cache."""
    bs = c["block"]
    pages = [-(-k // bs) for k in keys]
    blocks = sum(pages) + 8
    perm = torch.randperm(blocks, generator=_gen(seed, 2), device=DEV).to(torch.int32)
    rows = np.zeros((len(keys), max(pages)), dtype=np.int64)
    at = 0
    for i, p in enumerate(pages):
        rows[i, :p] = np.arange(at, at + p)
        at += p
    return perm[torch.from_numpy(rows).to(DEV)].contiguous(), blocks


def _batch(c, seed):
    q_lens, keys = _lens(c)
    table, blocks = _table(c, keys, seed)
    cu = np.concatenate([[0], np.cumsum(q_lens)]).astype(np.int32)
    s = {"q_lens": q_lens, "keys": keys, "cu_host": torch.from_numpy(cu), "blocks": blocks, "table": table,
         "cu": torch.from_numpy(cu).to(DEV), "lens": torch.tensor(keys, dtype=torch.int32, device=DEV)}
    s["q"] = torch.randn(int(cu[-1]), c["hq"], c["d"], generator=_gen(seed, 3), device=DEV, dtype=torch.bfloat16)
    s["out"] = torch.zeros_like(s["q"])
    short = [q for q in q_lens if q <= ck.SHORT_Q]
    s["segm"] = None
    if short and ck.split_pays(np.asarray(q_lens), np.asarray(keys), c["hkv"], ck.one_pass_fill(DEV)):
        s["segm"] = ck.split_buffers(sum(short), c["hq"], c["d"], ck.SPLIT_PIECES, DEV)
    return s


def _new_rows(c, n, gain, mu, g):
    k = torch.randn(n, c["hkv"], c["d"], generator=g, device=DEV) * gain + mu
    v = torch.randn(n, c["hkv"], c["d"], generator=g, device=DEV)
    return k.to(torch.bfloat16), v.to(torch.bfloat16)


# ------------------------------------------------------------------------------------------------ one case
def prepare(case, seed):
    c = dict(case)
    static, gain = _static(c, seed)
    if c["kind"] == "write":
        n, bs = c["tokens"], c["block"]
        blocks = -(-4 * n // bs)
        slots = torch.randperm(blocks * bs, generator=_gen(seed, 4), device=DEV)[:n]
        slots[torch.rand(n, generator=_gen(seed, 5), device=DEV) < c["pad"]] = -1
        kv = torch.zeros(_cache_shape(c, blocks), dtype=torch.int8, device=DEV)
        key, value = _new_rows(c, n, gain, static["k_mu"], _gen(seed, 6))
        kc, vc = _views(c, kv)
        return {"case": c, "static": static, "key": key, "value": value, "slots": slots, "kv": kv, "kc": kc, "vc": vc}
    s = _batch(c, seed)
    s.update(case=c, static=static, scale=c["d"] ** -0.5)
    if c["kind"] != "graph":
        s["kc"], s["vc"] = _views(c, _codes(_cache_shape(c, s["blocks"]), _gen(seed, 7)))
        s["plan"] = ck.plan_long(s["cu_host"], torch.tensor(s["keys"]), c["block"])
        return s
    # a decode step's layers: every layer its own cache, new K / V rows, q and output; the new token is
    # the last key of its request
    n, bs = c["requests"], c["block"]
    last = s["lens"].long() - 1
    s["slots"] = s["table"].gather(1, (last // bs)[:, None])[:, 0].long() * bs + last % bs
    s["segm"] = ck.split_buffers(n, c["hq"], c["d"], ck.SPLIT_PIECES, DEV)   # a captured call always carries them
    s["layers"] = []
    for k in range(c["layers"]):
        kv = _codes(_cache_shape(c, s["blocks"]), _gen(seed, 100 + k))
        key, value = _new_rows(c, n, gain, static["k_mu"], _gen(seed, 200 + k))
        q = torch.randn(n, c["hq"], c["d"], generator=_gen(seed, 300 + k), device=DEV, dtype=torch.bfloat16)
        kc, vc = _views(c, kv)
        s["layers"].append({"kv": kv, "kc": kc, "vc": vc, "key": key, "value": value, "q": q, "out": torch.zeros_like(q)})
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        _layers(s)
    torch.cuda.current_stream().wait_stream(side)
    s["graph"] = torch.cuda.CUDAGraph()
    with torch.cuda.graph(s["graph"]):
        _layers(s)
    return s


def _layers(s):
    for y in s["layers"]:
        ck.quant_reshape_and_cache(y["key"], y["value"], y["kc"], y["vc"], s["slots"], s["static"])
        ck.paged_attention(y["q"], y["kc"], y["vc"], y["out"], s["cu"], s["lens"], s["table"], 1, s["scale"],
                           s["static"], None, s["segm"])


def run(state):
    s = state
    kind = s["case"]["kind"]
    if kind == "write":
        ck.quant_reshape_and_cache(s["key"], s["value"], s["kc"], s["vc"], s["slots"], s["static"])
        return s["kv"]
    if kind == "graph":
        s["graph"].replay()
        return {"out": [y["out"] for y in s["layers"]], "cache": [y["kv"] for y in s["layers"]]}
    return ck.paged_attention(s["q"], s["kc"], s["vc"], s["out"], s["cu"], s["lens"], s["table"], max(s["q_lens"]),
                              s["scale"], s["static"], s["plan"], s["segm"])


def work(case):
    c = case
    hq, hkv, d = c["hq"], c["hkv"], c["d"]
    tables = 4 * hkv * ((2 * d if c["per_channel"] else 2) + d)
    if c["kind"] == "write":
        return {"bytes": c["tokens"] * (1 - c["pad"]) * hkv * d * 6 + 8 * c["tokens"] + tables, "flops": 0}
    q_lens, keys = _lens(c)
    pages = sum(-(-k // c["block"]) for k in keys)
    kv = sum(keys) * hkv * d * 2 + 4 * pages + 8 * len(keys)
    rows = sum(q_lens)
    pairs = sum(q * (k - q) + q * (q + 1) // 2 for q, k in zip(q_lens, keys))
    w = {"bytes": kv + rows * hq * d * 4 + tables, "flops": 4 * d * hq * pairs}
    if c["kind"] == "graph":
        w = {"bytes": c["layers"] * (w["bytes"] + rows * (hkv * d * 6 + 8)), "flops": c["layers"] * w["flops"]}
    return w


def tolerance(case):
    """Codes are exact. Measured against exact(): 1.6e-3 to 1.8e-3 for the INT8 attention (the bf16 output's
    rounding), 5e-3 to 8e-3 for the long-query path (K and V rounded to bf16 as well)."""
    if case["kind"] == "write":
        return "exact"
    return {"rel": 2e-2 if case["kind"] == "step" else 7e-3}


# ------------------------------------------------------------------------------------------------ 64 bits
def _quantize(x, scale):
    """The stored code: fp32 by definition (round half to even of the fp32 quotient, saturated)."""
    return torch.round(x / scale).clamp(-127, 127).to(torch.int8)


def _written(c, kv, key, value, slots, static):
    kc, vc = _views(c, kv)
    ok = (slots >= 0).nonzero()[:, 0]
    at = slots[ok]
    bs = c["block"]
    kc[at // bs, at % bs] = _quantize(key[ok].float() - static["k_mu"], static["k_scale"])
    vc[at // bs, at % bs] = _quantize(value[ok].float(), static["v_scale"])
    return kv


def _pages(cache, ids, n):
    """float64 [H, n, D] of a request's first n keys."""
    return cache[ids].flatten(0, 1)[:n].permute(1, 0, 2).double().contiguous()


def _short_exact(c, q, k, v, static, scale):
    """One short-query request in 64 bits: q [t, Hq, D] quantized with one fp32 scale per (token, head), the
    softmax's weights quantized per 32-key tile (the operator's definition), everything else exact."""
    hkv, d = c["hkv"], c["d"]
    t, hq = q.shape[:2]
    L = k.shape[1]
    ks = static["k_scale"]
    x = q.float().view(t, hkv, hq // hkv, d)
    if c["per_channel"]:
        x = x * ks[None, :, None]
    sq = (x.abs().amax(-1, keepdim=True) / 127).clamp_min(1e-8)
    codes = torch.round(x / sq).clamp(-127, 127).double()
    fac = sq.double() * (1.0 if c["per_channel"] else ks[None, :, None].double()) * scale
    out = torch.empty(t, hq, d, dtype=torch.float64, device=q.device)
    tiles = -(-L // 32)
    col = torch.arange(tiles * 32, device=q.device)
    for h in range(hkv):
        rows = codes[:, h].reshape(-1, d)
        s = torch.full((rows.shape[0], tiles * 32), -math.inf, dtype=torch.float64, device=q.device)
        s[:, :L] = (rows @ k[h].t()) * fac[:, h].reshape(-1, 1)
        lim = L - t + 1 + torch.arange(t, device=q.device).repeat_interleave(hq // hkv)
        s.masked_fill_(col[None] >= lim[:, None], -math.inf)
        p = torch.exp(s - s.amax(-1, keepdim=True)).view(rows.shape[0], tiles, 32)
        ps = (p.amax(-1, keepdim=True) / 127).clamp_min(1e-300)
        p = (torch.round(p / ps) * ps).view(rows.shape[0], -1)
        o = (p[:, :L] @ v[h]) / p.sum(-1, keepdim=True)
        out[:, h * (hq // hkv):(h + 1) * (hq // hkv)] = o.view(t, hq // hkv, d)
    return out * static["v_scale"].double().repeat_interleave(hq // hkv, 0)


def _long_exact(c, q, k, v, static, scale):
    """One long-query request in 64 bits: causal attention over code x scale."""
    hkv, d = c["hkv"], c["d"]
    t, hq = q.shape[:2]
    L, G = k.shape[1], hq // hkv
    out = torch.empty(t, hq, d, dtype=torch.float64, device=q.device)
    step = max(1, (1 << 26) // L)
    for h in range(hkv):
        kk = (k[h] * static["k_scale"][h].double()).t().contiguous()
        vv = v[h] * static["v_scale"][h].double()
        for g in range(G):
            for a in range(0, t, step):
                b = min(t, a + step)
                n = L - t + b                       # keys the last row of the block sees
                s = (q[a:b, h * G + g].double() @ kk[:, :n]) * scale
                lim = L - t + 1 + torch.arange(a, b, device=q.device)
                s.masked_fill_(torch.arange(n, device=q.device)[None] >= lim[:, None], -math.inf)
                out[a:b, h * G + g] = torch.softmax(s, -1) @ vv[:n]
    return out


def _attention_exact(c, s, q, kc, vc):
    out = []
    bs, at = c["block"], 0
    for r, (ql, n) in enumerate(zip(s["q_lens"], s["keys"])):
        ids = s["table"][r, :-(-n // bs)].long()
        one = _short_exact if ql <= ck.SHORT_Q else _long_exact
        out.append(one(c, q[at:at + ql], _pages(kc, ids, n), _pages(vc, ids, n), s["static"], s["scale"]))
        at += ql
    return torch.cat(out)


def exact(case, seed):
    c = dict(case)
    static, gain = _static(c, seed)
    s = prepare(case, seed)
    if c["kind"] == "write":
        return _written(c, s["kv"], s["key"], s["value"], s["slots"], static)
    if c["kind"] == "graph":
        cache = [_written(c, y["kv"], y["key"], y["value"], s["slots"], static) for y in s["layers"]]
        return {"out": [_attention_exact(c, s, y["q"], y["kc"], y["vc"]) for y in s["layers"]], "cache": cache}
    return _attention_exact(c, s, s["q"], s["kc"], s["vc"])
