"""The attention path's work as a serving engine has it done, one layer's call at a time.

A case is a dict of plain values:

* ``kind`` "attention": one ``Attention.forward`` (the new K/V rows stored, then attention over
  the paged cache). ``decode`` sequences bring one new token each over contexts of
  ``ctx_lo .. ctx_hi`` tokens; ``prompts`` sequences bring ``new_lo .. new_hi`` new tokens each
  over ``pre_lo .. pre_hi`` tokens that are cached already. A step of decode rows alone takes
  the decode kernel, any other step the variable-length one, as the engine's context says.
* ``kind`` "compress": one layer's compression step of ``topk`` sequences out of a batch, whose
  windows' tokens were stored since the step before (a step leaves the kept rows in their place).
* ``kind`` "norm_rope": q/k RMSNorm + RoPE + cache store of ``tokens`` tokens.

``hq``/``hk`` are the query and KV heads of one GPU (head_dim 128, blocks of 256 tokens), ``kv``
the cache's type (``bf16``, ``fp16``, ``fp8``); q and the outputs are bf16, or fp16 with an fp16
cache. ``shape`` seeds the lengths, so that a case's work does not depend on its inputs' seed.
"""
from __future__ import annotations

import importlib
import math
import random
from types import SimpleNamespace

import torch

nkv = importlib.import_module("nanokv-llm_amd")
compress_utils = importlib.import_module("nanokv-llm_amd.layers.compress_utils")

D = 128
BLOCK = 256
SCALE = D ** -0.5
WINDOW = 4            # blocks scored by a compression step
KEEP = 2 * BLOCK + 1  # tokens kept of them
MAX_POS = 40960
EPS = 1e-6
K_SCALE, V_SCALE = 0.02, 0.02  # fp8 pools: N(0, 1) rows within +-448 codes


def _attention(name, hq, hk, kv="bf16", decode=0, ctx_lo=0, ctx_hi=0, prompts=0, new_lo=0,
               new_hi=0, pre_lo=0, pre_hi=0, shape=1):
    c = dict(kind="attention", hq=hq, hk=hk, kv=kv, decode=decode, ctx_lo=ctx_lo, ctx_hi=ctx_hi,
             prompts=prompts, new_lo=new_lo, new_hi=new_hi, pre_lo=pre_lo, pre_hi=pre_hi,
             shape=shape)
    return dict(c, name=name) if name else c


def listed():
    return [
        # A few users on the smallest model: launches and latency.
        _attention("decode_4_short", 16, 8, decode=4, ctx_lo=300, ctx_hi=1000),
        # One user deep into a long conversation.
        _attention("decode_1_long", 32, 8, decode=1, ctx_lo=23001, ctx_hi=23001),
        # The benchmark's decode batch.
        _attention("decode_64", 32, 8, decode=64, ctx_lo=2048, ctx_hi=8192, shape=2),
        # High concurrency on half a model (two GPUs share it), fp8 pool, ragged contexts.
        _attention("decode_200_fp8", 16, 4, "fp8", decode=200, ctx_lo=100, ctx_hi=6000, shape=3),
        # Long contexts on the largest model.
        _attention("decode_96_long", 64, 8, decode=96, ctx_lo=1024, ctx_hi=16384, shape=4),
        # One short prompt, nothing else to run with it: time to first token.
        _attention("prompt_short", 16, 8, prompts=1, new_lo=333, new_hi=333),
        # The scheduler's 512-token share of one long prompt, late in that prompt.
        _attention("chunk_long_prefix", 32, 8, prompts=1, new_lo=512, new_hi=512, pre_lo=12288,
                   pre_hi=12288),
        # A step of continuous batching: decode rows run with two prompts' 512-token shares.
        _attention("mixed_step", 32, 8, decode=48, ctx_lo=300, ctx_hi=6000, prompts=2,
                   new_lo=512, new_hi=512, pre_lo=0, pre_hi=3072, shape=5),
        # A batch of whole prompts.
        _attention("prompts_16", 32, 8, prompts=16, new_lo=512, new_hi=4096, shape=6),
        # Large chunks of many prompts, the heaviest step.
        _attention("chunks_16", 32, 8, prompts=16, new_lo=2048, new_hi=2048, pre_lo=0,
                   pre_hi=8192, shape=7),
        # The periodic compression step of a batch of 500, one layer.
        dict(kind="compress", name="compress_20", hq=32, hk=8, kv="bf16", batch=500, topk=20,
             ctx_lo=1500, ctx_hi=4096, agg="group", shape=8),
        # Between the qkv projection and attention, a prefill step's tokens.
        dict(kind="norm_rope", name="norm_rope_9001", hq=32, hk=8, kv="bf16", tokens=9001),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    # (query heads, KV heads) of one GPU: whole models, and halves and quarters of them
    hq, hk = rng.choice([(16, 8), (32, 8), (64, 8), (40, 8), (16, 4), (32, 4), (8, 2), (16, 2)])
    kv = rng.choice(["bf16", "bf16", "bf16", "fp16", "fp8"])
    shape = rng.randrange(1 << 20)
    what = rng.choice(["decode", "decode", "decode", "prompt", "prompt", "mixed", "mixed",
                       "compress", "norm_rope"])
    if what == "decode":
        n = _log_int(rng, 1, 400)
        hi = _log_int(rng, 64, min(32768, 1_000_000 // n))
        lo = max(1, int(hi * rng.uniform(0.05, 1.0)))
        return _attention("", hq, hk, kv, decode=n, ctx_lo=lo, ctx_hi=hi, shape=shape)
    if what == "prompt":
        n = _log_int(rng, 1, 16)
        new_hi = _log_int(rng, 16, 3000)
        pre_hi = rng.choice([0, _log_int(rng, 100, 12000 if n <= 4 else 4096)])
        return _attention("", min(hq, 32), hk, kv, prompts=n,
                          new_lo=max(1, int(new_hi * rng.uniform(0.2, 1.0))), new_hi=new_hi,
                          pre_lo=int(pre_hi * rng.uniform(0.0, 1.0)), pre_hi=pre_hi, shape=shape)
    if what == "mixed":
        hi = _log_int(rng, 200, 8192)
        return _attention("", hq, hk, kv, decode=_log_int(rng, 1, 100),
                          ctx_lo=max(1, int(hi * rng.uniform(0.05, 1.0))), ctx_hi=hi,
                          prompts=rng.randint(1, 4), new_lo=rng.randint(1, 512), new_hi=512,
                          pre_lo=0, pre_hi=rng.choice([0, _log_int(rng, 100, 6000)]),
                          shape=shape)
    if what == "compress":
        batch = _log_int(rng, 8, 500)
        hi = _log_int(rng, 2048, 8192)
        return dict(kind="compress", hq=hq, hk=hk, kv=kv, batch=batch,
                    topk=rng.randint(1, min(batch, 24)), ctx_lo=1100, ctx_hi=hi,
                    agg=rng.choice(["group", "all"]), shape=shape)
    return dict(kind="norm_rope", hq=hq, hk=hk, kv=rng.choice(["bf16", "fp16"]),
                tokens=_log_int(rng, 1, 20000))


# ------------------------------------------------------------------ lengths and tables

def _lengths(rng, n, lo, hi):
    """n lengths of lo .. hi: uniform, or uniform in the logarithm over more than a factor 8."""
    if lo > 0 and hi > 8 * lo:
        return [_log_int(rng, lo, hi) for _ in range(n)]
    return [rng.randint(lo, hi) for _ in range(n)]


def _step_lengths(case):
    """(new tokens, keys) of each sequence: decode rows first, as the scheduler puts them."""
    rng = random.Random(case["shape"])
    ctx = _lengths(rng, case["decode"], case["ctx_lo"], case["ctx_hi"])
    new = _lengths(rng, case["prompts"], case["new_lo"], case["new_hi"])
    pre = _lengths(rng, case["prompts"], case["pre_lo"], case["pre_hi"])
    return [1] * len(ctx) + new, ctx + [a + b for a, b in zip(new, pre)]


def _compress_lengths(case):
    """Lengths of the batch, and the topk longest that are eligible, in batch order."""
    rng = random.Random(case["shape"])
    lens = _lengths(rng, case["batch"], case["ctx_lo"], case["ctx_hi"])
    fit = [i for i, n in enumerate(lens) if n % BLOCK != BLOCK - 1]
    chosen = sorted(sorted(fit, key=lambda i: (-lens[i], i))[:case["topk"]])
    return lens, chosen


def _tables(lens, gen):
    """Block tables over a pool in random order, padded with -1, and the pool's blocks."""
    need = [-(-n // BLOCK) for n in lens]
    pool = sum(need) + 8
    ids = torch.randperm(pool, generator=gen, dtype=torch.int32)
    table = torch.full((len(lens), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        table[i, :n] = ids[at:at + n]
        at += n
    return table, pool


def _dtype(case):
    return torch.float16 if case["kv"] == "fp16" else torch.bfloat16


def _caches(case, pool, gen):
    """K and V as the two halves of one pool; fp8 pools hold codes of N(0, 1) / scale."""
    shape = (2, pool, BLOCK, case["hk"], D)
    kv = torch.randn(shape, generator=gen, device="cuda", dtype=_dtype(case))
    if case["kv"] == "fp8":
        kv[0].div_(K_SCALE)
        kv[1].div_(V_SCALE)
        kv = kv.to(torch.float8_e4m3fn)
    return kv[0], kv[1]


def _whole(cache):
    """A cache as an output: fp8 codes as bytes."""
    return cache.view(torch.uint8) if cache.dtype == torch.float8_e4m3fn else cache


# ------------------------------------------------------------------ prepare and run

def prepare(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed * 2 + 1)
    host = torch.Generator().manual_seed(seed * 2 + 1)
    return _PREPARE[case["kind"]](case, gen, host)


def _randn(gen, *shape, dtype, scale=1.0):
    return (torch.randn(shape, generator=gen, device="cuda", dtype=torch.float32) * scale).to(dtype)


def _prepare_attention(case, gen, host):
    new, keys = _step_lengths(case)
    table, pool = _tables(keys, host)
    hq, hk, dt = case["hq"], case["hk"], _dtype(case)
    k_cache, v_cache = _caches(case, pool, gen)
    layer = nkv.Attention(hq, D, SCALE, hk, SimpleNamespace(kv_compress_enabled=False), 1)
    layer.k_cache, layer.v_cache = k_cache, v_cache
    if case["kv"] == "fp8":
        layer.k_scale, layer.v_scale = K_SCALE, V_SCALE
    n = sum(new)
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    pos = torch.cat([torch.arange(b - a, b) for a, b in zip(new, keys)])
    slots = (table[seq, pos // BLOCK].long() * BLOCK + pos % BLOCK).to(torch.int32)
    sums = lambda v: torch.tensor([0] + v, dtype=torch.int32).cumsum(0, dtype=torch.int32)  # noqa: E731
    return dict(
        kind="attention", layer=layer, decode_only=case["prompts"] == 0,
        q=_randn(gen, n, hq, D, dtype=dt, scale=2.0), k=_randn(gen, n, hk, D, dtype=dt),
        v=_randn(gen, n, hk, D, dtype=dt), slots=slots.cuda(), table=table.cuda(),
        lens=torch.tensor(keys, dtype=torch.int32).cuda(), cu_q=sums(new).cuda(),
        cu_k=sums(keys).cuda(), max_q=max(new), max_k=max(keys),
        caches=(_whole(k_cache), _whole(v_cache)), new=new, keys=keys)


def _run_attention(s):
    if s["decode_only"]:
        nkv.set_context(True, slot_mapping=s["slots"], context_lens=s["lens"],
                        block_tables=s["table"])
    else:
        nkv.set_context(False, s["cu_q"], s["cu_k"], s["max_q"], s["max_k"], s["slots"],
                        s["lens"], s["table"])
    return dict(out=s["layer"](s["q"], s["k"], s["v"], 0), k_cache=s["caches"][0],
                v_cache=s["caches"][1])


def _prepare_compress(case, gen, host):
    lens, chosen = _compress_lengths(case)
    # only the chosen sequences' blocks are touched: the others own one each here
    table, pool = _tables([n if i in set(chosen) else 1 for i, n in enumerate(lens)], host)
    pos = [(lens[i] // BLOCK - WINDOW) * BLOCK + torch.arange(WINDOW * BLOCK) for i in chosen]
    slots = torch.cat([table[i, p // BLOCK].long() * BLOCK + p % BLOCK
                       for i, p in zip(chosen, pos)]).to(torch.int32)
    hq, hk, m = case["hq"], case["hk"], len(chosen)
    sets, cand = (1 if case["agg"] == "all" else hk), WINDOW * BLOCK - 1
    k_cache, v_cache = _caches(case, pool, gen)
    base = torch.tensor(lens, dtype=torch.int32).cuda()
    need = compress_utils.select_workspace_bytes(m, hq, hk, WINDOW, BLOCK)
    return dict(
        kind="compress", agg=case["agg"], k_scale=K_SCALE if case["kv"] == "fp8" else 1.0,
        v_scale=V_SCALE if case["kv"] == "fp8" else 1.0, slots=slots.cuda(),
        k=_randn(gen, slots.numel(), hk, D, dtype=_dtype(case)),
        v=_randn(gen, slots.numel(), hk, D, dtype=_dtype(case)),
        q=_randn(gen, len(lens), hq, D, dtype=_dtype(case), scale=2.0), k_cache=k_cache,
        v_cache=v_cache, table=table.cuda(), base=base, lens=base.clone(),
        chosen=torch.tensor(chosen, dtype=torch.int32).cuda(),
        importance=torch.empty(m, sets, cand, dtype=torch.float32, device="cuda"),
        keep=torch.empty(m, sets, KEEP, dtype=torch.int32, device="cuda"),
        workspace=torch.empty(max(need, 4), dtype=torch.uint8, device="cuda"),
        caches=(_whole(k_cache), _whole(v_cache)))


def _run_compress(s):
    nkv.store_kvcache(s["k"], s["v"], s["k_cache"], s["v_cache"], s["slots"], s["k_scale"],
                      s["v_scale"])
    keep, importance = compress_utils.compress_step(
        s["q"], s["k_cache"], s["v_cache"], s["table"], s["base"], s["lens"], s["chosen"],
        WINDOW, KEEP, SCALE, s["agg"], importance=s["importance"], keep_idx=s["keep"],
        workspace=s["workspace"], k_scale=s["k_scale"])
    return dict(importance=importance, keep=keep, lens=s["lens"], k_cache=s["caches"][0],
                v_cache=s["caches"][1])


def _rope_table():
    inv = 1.0 / (1e6 ** (torch.arange(0, D, 2, dtype=torch.float64) / D))
    a = torch.arange(MAX_POS, dtype=torch.float64)[:, None] * inv
    return torch.cat([a.cos(), a.sin()], dim=-1).float()


_ROPE = []  # the rotary table, which a model makes once


def _prepare_norm_rope(case, gen, host):
    if not _ROPE:
        _ROPE.append(_rope_table().cuda())
    n, hq, hk, dt = case["tokens"], case["hq"], case["hk"], _dtype(case)
    pool = -(-n // BLOCK) + 8
    qkv = _randn(gen, n, (hq + 2 * hk) * D, dtype=dt)
    slots = torch.randperm(pool * BLOCK, generator=host, dtype=torch.int32)[:n]
    pos = torch.randint(0, MAX_POS, (n,), generator=host)
    k_cache = torch.zeros(pool, BLOCK, hk, D, dtype=dt, device="cuda")
    return dict(
        kind="norm_rope", q=qkv[:, :hq * D].view(n, hq, D),
        k=qkv[:, hq * D:(hq + hk) * D].view(n, hk, D), v=qkv[:, (hq + hk) * D:].view(n, hk, D),
        pos=pos.cuda(), qw=_randn(gen, D, dtype=dt, scale=0.2) + 1,
        kw=_randn(gen, D, dtype=dt, scale=0.2) + 1, table=_ROPE[0], k_cache=k_cache,
        v_cache=torch.zeros_like(k_cache), slots=slots.cuda())


def _run_norm_rope(s):
    q, _, _ = nkv.qk_norm_rope_store(s["pos"], s["q"], s["k"], s["v"], s["table"], s["qw"],
                                     s["kw"], EPS, k_cache=s["k_cache"], v_cache=s["v_cache"],
                                     slot_mapping=s["slots"], need_k=False)
    return dict(q=q, k_cache=s["k_cache"], v_cache=s["v_cache"])


_PREPARE = {"attention": _prepare_attention, "compress": _prepare_compress,
            "norm_rope": _prepare_norm_rope}
_RUN = {"attention": _run_attention, "compress": _run_compress, "norm_rope": _run_norm_rope}


def run(state):
    return _RUN[state["kind"]](state)


# ------------------------------------------------------------------ work

def work(case):
    hq, hk = case["hq"], case["hk"]
    el = 1 if case["kv"] == "fp8" else 2  # bytes of a cached value
    row = hk * D * el                     # of a token's K (or V) in the cache
    if case["kind"] == "attention":
        new, keys = _step_lengths(case)
        n = sum(new)
        pairs = sum(a * (b - a) + a * (a + 1) // 2 for a, b in zip(new, keys))
        # cached rows read (the new ones among them), new rows read and stored, q and out,
        # slots and tables
        return dict(bytes=2 * sum(keys) * row + 2 * n * hk * D * 2 + 2 * n * row
                    + 2 * n * hq * D * 2 + 4 * n + 4 * sum(-(-b // BLOCK) for b in keys),
                    flops=4 * hq * D * pairs)
    if case["kind"] == "compress":
        lens, chosen = _compress_lengths(case)
        m, tails = len(chosen), sum(lens[i] % BLOCK for i in chosen)
        # the windows' new rows read and stored; the windows' K, the kept V and the tails read;
        # kept and tail rows written; q
        stored = 2 * m * WINDOW * BLOCK
        read = m * (WINDOW * BLOCK + KEEP) + 2 * tails
        written = 2 * (m * KEEP + tails)
        return dict(bytes=stored * (hk * D * 2 + row) + (read + written) * row + m * hq * D * 2,
                    flops=2 * m * hq * D * WINDOW * BLOCK)
    n = case["tokens"]
    heads = hq + 2 * hk
    return dict(bytes=2 * n * heads * D * 2 + n * (D * 4 + 8 + 4), flops=n * (hq + hk) * D * 10)


# ------------------------------------------------------------------ tolerance and exact

def tolerance(case):
    if case["kind"] == "compress":
        # importance in 32 bits; kept sets, and with them the compacted caches, whole
        return {"rel": 1e-5, "max": 1e-4}
    # 16-bit outputs (each side about 1.8e-3 off 64 bits in bf16, an eighth of it in fp16), with
    # weights rounded to 16 bits for the second product
    if case["kv"] == "fp16":
        return {"rel": 1.5e-3, "max": 1e-2}
    return {"rel": 1e-2, "max": 6e-2}


def exact(case, seed):
    return _EXACT[case["kind"]](case, prepare(case, seed))


def _values(cache, scale, fp8):
    return cache.double() * (scale if fp8 else 1.0)


def _stored(s, kc, vc, hk, fp8):
    """The new K/V rows in their slots of the caches."""
    rows = s["slots"].long()
    for cache, x, scale in ((kc, s["k"], K_SCALE), (vc, s["v"], V_SCALE)):
        if fp8:
            x = (x.float() * (1.0 / scale)).clamp(-448, 448).to(torch.float8_e4m3fn)
        _whole(cache).view(-1, hk * D)[rows] = _whole(x).view(-1, hk * D)


def _exact_attention(case, s):
    fp8 = case["kv"] == "fp8"
    hq, hk = case["hq"], case["hk"]
    g = hq // hk
    kc, vc = s["layer"].k_cache, s["layer"].v_cache
    _stored(s, kc, vc, hk, fp8)
    out = torch.empty(sum(s["new"]), hq, D, dtype=torch.float64, device="cuda")
    at = 0
    for i, (lq, lk) in enumerate(zip(s["new"], s["keys"])):
        ids = s["table"][i, :-(-lk // BLOCK)].long()
        # whole blocks by bytes or 16-bit words (fp8 tensors cannot be indexed everywhere)
        k = _whole(kc)[ids].view(kc.dtype).reshape(-1, hk, D)[:lk]
        v = _whole(vc)[ids].view(vc.dtype).reshape(-1, hk, D)[:lk]
        key = torch.arange(lk, device="cuda")
        for h in range(hk):
            kh, vh = _values(k[:, h], K_SCALE, fp8), _values(v[:, h], V_SCALE, fp8)
            for j in range(0, lq, 1024):
                n = min(1024, lq - j)
                q = s["q"][at + j:at + j + n, h * g:(h + 1) * g].double().reshape(n * g, D)
                w = (q @ kh.t()) * SCALE
                last = lk - lq + j + torch.arange(n, device="cuda").repeat_interleave(g)
                w.masked_fill_(key[None, :] > last[:, None], -math.inf)
                out[at + j:at + j + n, h * g:(h + 1) * g] = (
                    torch.softmax(w, dim=-1) @ vh).view(n, g, D)
        at += lq
    return dict(out=out.unsqueeze(1) if s["decode_only"] else out, k_cache=s["caches"][0],
                v_cache=s["caches"][1])


def _exact_compress(case, s):
    fp8 = case["kv"] == "fp8"
    hq, hk = case["hq"], case["hk"]
    g, w = hq // hk, WINDOW * BLOCK
    lens, chosen = _compress_lengths(case)
    _stored(s, s["k_cache"], s["v_cache"], hk, fp8)
    importance = torch.empty(len(chosen), hk, w - 1, dtype=torch.float64, device="cuda")
    for j, i in enumerate(chosen):
        full = lens[i] // BLOCK
        ids = s["table"][i, full - WINDOW:full].long()
        k = _values(_whole(s["k_cache"])[ids].view(s["k_cache"].dtype).reshape(w, hk, D),
                    K_SCALE, fp8)
        for h in range(hk):
            a = (s["q"][i, h * g:(h + 1) * g].double() @ k[:w - 1, h].t()) * SCALE
            a[:, 0] = -math.inf  # the first key is kept in any case and takes no weight
            importance[j, h] = torch.softmax(a, dim=-1).sum(0)
    if case["agg"] == "all":
        importance = importance.sum(1, keepdim=True)
    return dict(importance=importance, keep=None, lens=None, k_cache=None, v_cache=None)


def _exact_norm_rope(case, s):
    hk = case["hk"]
    cos, sin = s["table"].double()[s["pos"]].unsqueeze(1).chunk(2, dim=-1)

    def turned(x, w):
        x = x.double()
        x = x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()
        a, b = x.chunk(2, dim=-1)
        return torch.cat([a * cos - b * sin, b * cos + a * sin], dim=-1)

    rows = s["slots"].long()
    k_cache, v_cache = s["k_cache"].double(), s["v_cache"].double()
    k_cache.view(-1, hk, D)[rows] = turned(s["k"], s["kw"])
    v_cache.view(-1, hk, D)[rows] = s["v"].double()
    return dict(q=turned(s["q"], s["qw"]), k_cache=k_cache, v_cache=v_cache)


_EXACT = {"attention": _exact_attention, "compress": _exact_compress,
          "norm_rope": _exact_norm_rope}
