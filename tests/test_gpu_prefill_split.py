"""Variable-length attention with the keys split over the chip (nkv_prefill_varlen_split)
against the fp32 oracle: every form the entry point takes, at lengths around the edges of
tiles, key steps and ranges, and the launch rule's choice through Attention.forward."""
import importlib
from types import SimpleNamespace

import pytest
import torch

from oracle.attention_ref import varlen_prefill_ref

L = importlib.import_module("nanokv-llm_amd._lib")
TOL = 2e-2  # the repository's bar for 16-bit outputs of N(0, 1) values

# (new tokens, keys) per sequence
MIXES = {
    # decode rows, empty sequences, rows that see no key, one chunk on a prefix
    "mixed": [(1, 900), (0, 0), (1, 1), (0, 70), (49, 333), (1, 1500), (17, 9), (1, 64)],
    # one row whose keys every range shares
    "one_row": [(1, 2999)],
    # tiles of 48 queries at G = 4: one short of, at and one past a tile and a key step
    "edges": [(47, 63), (48, 64), (49, 65), (96, 128), (97, 1281)],
    # a sequence per range and more than one batch of 64 sequences
    "many": [(1 + i % 3, 30 * (i % 7) + 3) for i in range(130)],
    # decode rows alone, more than one batch of 64 of them
    "rows": [(1, 17 * (i % 40) + 1) for i in range(90)],
    # one chunk on a long prefix
    "chunk": [(130, 2311)],
}


def _inputs(dev, mix, Hq, Hk, D, kind, B, paged, seed):
    g = torch.Generator().manual_seed(seed)
    dt = torch.float16 if kind == "fp16" else torch.bfloat16
    lq, lk = [a for a, _ in mix], [b for _, b in mix]
    cs = lambda x: torch.tensor([0] + x).cumsum(0).to(torch.int32)  # noqa: E731
    q = torch.randn(sum(lq), Hq, D, generator=g).to(dt)
    if not paged:  # V a strided view, as of a qkv projection
        k = torch.randn(sum(lk), Hk, D, generator=g).to(dt)
        v = torch.randn(sum(lk), 3 * Hk, D, generator=g).to(dt)[:, Hk:2 * Hk]
        return q, k, v, cs(lq), cs(lk), None
    need = [-(-n // B) for n in lk]
    ids = torch.randperm(sum(need) + 3, generator=g).to(torch.int32)
    bt = torch.full((len(mix), max(need)), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = ids[at:at + n]
        at += n
    kv = torch.randn(2, sum(need) + 3, B, Hk, D, generator=g)
    kv = (kv * 16).to(torch.float8_e4m3fn) if kind == "fp8" else kv.to(dt)
    return q, kv[0], kv[1], cs(lq), cs(lk), bt


def _split(dev, q, k, v, cu_q, cu_k, bt, kind, scale, used=None, scales=None):
    N, Hq, D = q.shape
    t = {"bf16": L.NKV_KV_BF16, "fp16": L.NKV_KV_F16, "fp8": L.NKV_KV_FP8}[kind]
    Hk = k.size(-2)
    n_rows = k.size(0) * (k.size(1) if bt is not None else 1)
    ks, vs = (k.stride(0), v.stride(0)) if bt is None else (Hk * D, Hk * D)
    s = scales or (1 / 16 if kind == "fp8" else 1.0)
    d = [x.to(dev) if x is not None else None for x in (q, k, cu_q, cu_k, bt)]
    # a strided V stays strided on the device
    vd = v.to(dev) if v.is_contiguous() else \
        torch.empty_strided(v.shape, v.stride(), dtype=v.dtype, device=dev).copy_(v)
    nbytes = L.lib().nkv_prefill_split_workspace_bytes(cu_q.numel() - 1, Hq, Hk, D, t)
    ws = torch.full((nbytes,), 0xff, dtype=torch.uint8, device=dev)  # NaN where nothing is written
    out = torch.full((N, Hq, D), float("nan"), dtype=q.dtype, device=dev)
    max_q = int((cu_q[1:] - cu_q[:-1]).max())
    L.check(L.lib().nkv_prefill_varlen_split(
        t, d[0].data_ptr(), q.stride(0), d[1].data_ptr(), vd.data_ptr(), ks, vs,
        d[2].data_ptr(), d[3].data_ptr(), d[4].data_ptr() if bt is not None else None,
        bt.stride(0) if bt is not None else 0, bt.size(1) if bt is not None else 0,
        cu_q.numel() - 1, max_q, Hq, Hk, D, k.size(1) if bt is not None else 0, n_rows, scale,
        s, s, out.data_ptr(), out.stride(0), ws.data_ptr(), ws.numel(), L.stream_of(d[0])),
        "prefill_varlen_split")
    torch.cuda.synchronize()
    if used is not None:
        used.append(bool((ws != 0xff).any()))
    return out


@pytest.mark.gpu
@pytest.mark.parametrize("mix,Hq,Hk,D,kind,B,paged", [
    ("mixed", 32, 8, 128, "bf16", 256, True),
    ("mixed", 20, 4, 128, "fp16", 16, True),    # a group that leaves spare rows; 4 blocks a step
    ("mixed", 16, 2, 128, "fp8", 64, True),
    ("mixed", 16, 8, 128, "bf16", 0, False),
    ("mixed", 8, 4, 64, "bf16", 256, True),
    ("mixed", 8, 2, 256, "fp16", 64, True),
    ("mixed", 16, 4, 64, "fp8", 64, True),
    ("mixed", 4, 2, 256, "fp8", 256, True),
    ("mixed", 64, 1, 128, "bf16", 256, True),   # a group of 64: three queries a tile
    ("one_row", 32, 8, 128, "bf16", 256, True),
    ("one_row", 5, 1, 128, "fp8", 256, True),   # every range one part
    ("edges", 32, 8, 128, "bf16", 64, True),
    ("edges", 32, 8, 128, "fp16", 0, False),
    ("many", 8, 4, 128, "bf16", 16, True),
    ("many", 8, 2, 128, "fp8", 64, True),
    ("rows", 32, 8, 128, "bf16", 256, True),
    ("rows", 24, 1, 128, "fp16", 16, True),     # two column groups of query heads
    ("rows", 8, 4, 64, "bf16", 64, True),
    ("chunk", 32, 8, 128, "bf16", 256, True),
    ("chunk", 8, 1, 64, "fp16", 0, False),
])
def test_split_matches_the_oracle(dev, mix, Hq, Hk, D, kind, B, paged):
    print(mix, Hq, Hk, D, kind, B, paged, flush=True)
    q, k, v, cu_q, cu_k, bt = _inputs(dev, MIXES[mix], Hq, Hk, D, kind, B, paged, seed=5)
    out = _split(dev, q, k, v, cu_q, cu_k, bt, kind, D ** -0.5)
    s = 1 / 16 if kind == "fp8" else 1.0
    ref = varlen_prefill_ref(q.float(), k.float() * s, v.float() * s, cu_q, cu_k, D ** -0.5,
                             block_tables=bt)
    assert (out.float().cpu() - ref).abs().max().item() <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("rows", [[1], [16], [17], [32], [33], [1, 2], [16, 16], [0, 1, 0]])
@pytest.mark.parametrize("chunk", [None, (130, 2311)])
def test_split_computes_the_fewest_short_decode_rows(dev, kind, rows, chunk):
    """Decode rows of a chunk or two of keys, beside a chunk on a long prefix and alone: a
    vanishing share of the work, which still has its workgroups."""
    print(kind, rows, chunk, flush=True)
    mix = [(1, n) for n in rows] + ([chunk] if chunk else [])
    q, k, v, cu_q, cu_k, bt = _inputs(dev, mix, 32, 8, 128, kind, 256, True, seed=12)
    out = _split(dev, q, k, v, cu_q, cu_k, bt, kind, 128 ** -0.5)
    s = 1 / 16 if kind == "fp8" else 1.0
    ref = varlen_prefill_ref(q.float(), k.float() * s, v.float() * s, cu_q, cu_k, 128 ** -0.5,
                             block_tables=bt)
    assert (out.float().cpu() - ref).abs().max().item() <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("kind,Hq,Hk,D", [
    ("bf16", 65, 1, 128), ("bf16", 72, 1, 64), ("fp16", 128, 1, 128), ("fp8", 128, 1, 128),
    ("bf16", 256, 2, 128),
    # 256 (and 512) KV heads: two workgroups (one) each, fewer than a group of 80 needs
    ("bf16", 80 * 256, 256, 64), ("fp8", 2 * 512, 512, 64)])
@pytest.mark.parametrize("mix", [[(1, 200), (40, 1200)], [(40, 1200), (1, 1), (1, 17)],
                                 [(1, 40), (1, 700)]])
def test_split_gives_every_column_group_of_the_rows_a_wave(dev, kind, Hq, Hk, D, mix):
    """Groups of more than 64 query heads take more waves a row than a workgroup has."""
    if Hk > 2:
        mix = [(min(a, 3), min(b, 80)) for a, b in mix]
    print(kind, Hq, Hk, D, mix, flush=True)
    q, k, v, cu_q, cu_k, bt = _inputs(dev, mix, Hq, Hk, D, kind, 64, True, seed=14)
    out = _split(dev, q, k, v, cu_q, cu_k, bt, kind, D ** -0.5)
    s = 1 / 16 if kind == "fp8" else 1.0
    ref = varlen_prefill_ref(q.float(), k.float() * s, v.float() * s, cu_q, cu_k, D ** -0.5,
                             block_tables=bt)
    assert (out.float().cpu() - ref).abs().max().item() <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_attention_beside_a_long_chunk_keeps_a_new_sequences_row(nkv, dev, kind):
    """A step of a chunk late in a long prompt and the first decode step of a short one, through
    Attention.forward, whose plan takes the split launch for it."""
    mix = [(130, 4000), (1, 9)]
    q, k, v, cu_q, cu_k, bt = _inputs(dev, mix, 32, 8, 128, kind, 256, True, seed=13)
    t = L.NKV_KV_FP8 if kind == "fp8" else L.NKV_KV_BF16
    assert L.lib().nkv_prefill_split_plan(2, 131, 130, 4000, 32, 8, 128, t) > 0
    layer = nkv.Attention(32, 128, 128 ** -0.5, 8, SimpleNamespace(kv_compress_enabled=False), 1)
    layer.k_cache, layer.v_cache = k.to(dev), v.to(dev)
    s = layer.k_scale = layer.v_scale = 1 / 16 if kind == "fp8" else 1.0
    nkv.set_context(False, cu_q.to(dev), cu_k.to(dev), 130, 4000, None, None, bt.to(dev))
    out = layer(q.to(dev), None, None, 0, kv_stored=True)
    nkv.reset_context()
    ref = varlen_prefill_ref(q.float(), k.float() * s, v.float() * s, cu_q, cu_k, 128 ** -0.5,
                             block_tables=bt)
    assert (out.float().cpu() - ref).abs().max().item() <= TOL


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp8"])
def test_split_takes_invalid_blocks_as_zero_keys(nkv, dev, kind):
    """Table entries outside the pool, and keys past the table's width, are zero keys that take
    their weight, in the decode rows' stream too: the plain launch's results (two orders of
    the same sums, outputs rounded to bf16: 2^-8 of |out| < 4)."""
    mix = [(1, 700), (1, 300), (60, 500), (1, 200)]
    q, k, v, cu_q, cu_k, bt = _inputs(dev, mix, 16, 4, 128, kind, 64, True, seed=8)
    bt[0, 3], bt[1, 0], bt[2, 2], bt[3, 1] = -1, 10 ** 6, -7, -1
    bt = bt[:, :10].contiguous()  # row 0's last key block is past the table
    out = _split(dev, q, k, v, cu_q, cu_k, bt, kind, 128 ** -0.5)
    s = 1 / 16 if kind == "fp8" else 1.0
    plain = nkv.varlen_prefill(*(x.to(dev) for x in (q, k, v, cu_q, cu_k)), 60, 128 ** -0.5,
                               block_tables=bt.to(dev), k_scale=s, v_scale=s)
    assert (out.float() - plain.float()).abs().max().item() <= 2 ** -6


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("prompt", [None, (60, 500)])
def test_split_weighs_every_key_past_a_narrow_table(nkv, dev, kind, prompt):
    """Decode rows of up to 30000 keys over a table of 160: the keys past it are zeros that take
    their weight, all of them, however many ranges they would have made (the plain launch's
    results from two orders of the same sums: a bf16 ulp, 2^-6 where 2 <= |out| < 4, as the row
    of 160 keys with these peaked scores has)."""
    mix = [(1, 30000), (1, 9000), (1, 161), (1, 160)] + ([prompt] if prompt else [])
    g = torch.Generator().manual_seed(16)
    q, k, v, cu_q, cu_k, bt = _inputs(dev, [(a, min(b, 160)) for a, b in mix[:4]] + mix[4:],
                                      16, 4, 128, kind, 16, True, seed=16)
    q = (3 * torch.randn(q.shape, generator=g)).to(q.dtype)  # the keys there weigh as much
    cu_k = torch.tensor([0] + [b for _, b in mix]).cumsum(0).to(torch.int32)
    bt = bt[:, :10].contiguous()
    out = _split(dev, q, k, v, cu_q, cu_k, bt, kind, 128 ** -0.5)
    s = 1 / 16 if kind == "fp8" else 1.0
    max_q = 60 if prompt else 1
    plain = nkv.varlen_prefill(*(x.to(dev) for x in (q, k, v, cu_q, cu_k)), max_q, 128 ** -0.5,
                               block_tables=bt.to(dev), k_scale=s, v_scale=s)
    assert (out.float() - plain.float()).abs().max().item() <= 2 ** -6


@pytest.mark.gpu
@pytest.mark.parametrize("kind,scales", [("bf16", 3.0), ("fp16", -1.0)])
def test_split_uses_the_scales_of_an_fp8_pool_only(dev, kind, scales):
    """Finished tiles, merged ones and decode rows alike."""
    q, k, v, cu_q, cu_k, bt = _inputs(dev, MIXES["mixed"], 16, 4, 128, kind, 64, True, seed=17)
    args = (dev, q, k, v, cu_q, cu_k, bt, kind, 128 ** -0.5)
    assert torch.equal(_split(*args, scales=scales), _split(*args))


@pytest.mark.gpu
@pytest.mark.parametrize("width,split", [(16, True), (5 << 20, False)])
def test_split_leaves_tables_beyond_32_bit_positions_to_the_plain_launch(nkv, dev, width, split):
    """A table whose rows could hold more keys than positions (1.3e9 of 256 blocks): the plain
    launch's own bits, and the workspace not touched."""
    q, k, v, cu_q, cu_k, bt = _inputs(dev, [(200, 900), (1, 40)], 8, 4, 128, "bf16", 256, True,
                                      seed=15)
    wide = torch.full((2, width), -1, dtype=torch.int32)
    wide[:, :bt.size(1)] = bt
    used = []
    out = _split(dev, q, k, v, cu_q, cu_k, wide, "bf16", 128 ** -0.5, used)
    plain = nkv.varlen_prefill(*(x.to(dev) for x in (q, k, v, cu_q, cu_k)), 200, 128 ** -0.5,
                               block_tables=bt.to(dev))
    assert used == [split] and torch.equal(out, plain) == (not split)
    assert (out.float() - plain.float()).abs().max().item() <= 2 ** -7  # |out| < 2: half an ulp


@pytest.mark.gpu
def test_attention_takes_a_long_prefix_to_the_split_launch(nkv, dev):
    """Attention.forward against the plain launch: two orders of the same sums, each weight
    and output rounded to bf16 (2^-8 relative, |out| < 1 here); then captured in a graph and
    replayed over other queries, with eager work between the replays."""
    mix = [(130, 9000), (1, 400)]
    q, k, v, cu_q, cu_k, bt = (x.to(dev) for x in
                               _inputs(dev, mix, 32, 8, 128, "bf16", 256, True, seed=6))
    assert L.lib().nkv_prefill_split_plan(2, 131, 130, 9000, 32, 8, 128, L.NKV_KV_BF16) > 0
    layer = nkv.Attention(32, 128, 128 ** -0.5, 8, SimpleNamespace(kv_compress_enabled=False), 1)
    layer.k_cache, layer.v_cache = k, v
    nkv.set_context(False, cu_q, cu_k, 130, 9000, None, None, bt)
    run = lambda: layer(q, None, None, 0, kv_stored=True)  # noqa: E731
    plain = lambda: nkv.varlen_prefill(q, k, v, cu_q, cu_k, 130, 128 ** -0.5,  # noqa: E731
                                       block_tables=bt)
    assert (run().float() - plain().float()).abs().max().item() <= 2 ** -8
    stream = torch.cuda.Stream()
    with torch.cuda.stream(stream):
        run()
    stream.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph, stream=stream):
        out = run()
    for scale in (1.0, -0.5, 2.0):
        q.mul_(scale)
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, run())
    nkv.reset_context()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,Hq,Hk,D", [("bf16", 32, 8, 128), ("fp16", 20, 4, 128),
                                          ("fp8", 16, 2, 128), ("bf16", 8, 2, 64),
                                          ("bf16", 128, 1, 128)])
@pytest.mark.parametrize("n", [1, 30, 70])
def test_plain_tile_sizes_match_the_oracle(nkv, dev, kind, Hq, Hk, D, n):
    """Plain launches of one, two and three row groups a wave: the first sequences' lengths stand
    at the edges of their tiles, the others fill up to the workgroups that change the size."""
    g = Hq // Hk
    mix = [(max(1, 64 * rg // g + d), 70 * rg + d) for rg in (1, 2, 3) for d in (-1, 0, 1)]
    mix = [(min(a, b), b) for a, b in mix][:9] + [(400, 400)] * (n > 1) + [(250, 300)] * (n - 1)
    q, k, v, cu_q, cu_k, bt = _inputs(dev, mix, Hq, Hk, D, kind, 64, True, seed=11)
    s = 1 / 16 if kind == "fp8" else 1.0
    out = nkv.varlen_prefill(*(x.to(dev) for x in (q, k, v, cu_q, cu_k)),
                             max(a for a, _ in mix), D ** -0.5, block_tables=bt.to(dev),
                             k_scale=s, v_scale=s)
    torch.cuda.synchronize()
    some = 10  # sequences compared
    ref = varlen_prefill_ref(q[:int(cu_q[some - 1])].float(), k.float() * s, v.float() * s,
                             cu_q[:some], cu_k[:some], D ** -0.5, block_tables=bt[:some - 1])
    assert (out[:ref.size(0)].float().cpu() - ref).abs().max().item() <= TOL
    assert bool(torch.isfinite(out.float()).all())


# (sequences, rows of q, longest new and key lengths, Hq, Hk, head_dim, kv_type): split launches
# measured at 0.55 of the plain one's time or less
SPLIT_FASTER = [(40, 135, 96, 2203, 32, 8, 256, 0), (1, 10, 10, 1748, 8, 8, 256, 2),
                (40, 54, 15, 6000, 128, 2, 128, 2), (1, 5, 5, 3255, 48, 1, 256, 0),
                (2, 95, 85, 11968, 28, 4, 256, 2)]


def test_split_plan_and_arguments_on_the_host():
    """The rule, and what the entry point refuses, without a GPU."""
    lib = L.lib()
    plan = lambda *a: lib.nkv_prefill_split_plan(*a)  # noqa: E731
    size = lambda n: lib.nkv_prefill_split_workspace_bytes(n, 32, 8, 128, L.NKV_KV_BF16)  # noqa: E731
    full = size(1)
    assert plan(1, 512, 512, 12800, 32, 8, 128, L.NKV_KV_BF16) == full > 0
    assert plan(50, 1072, 512, 5700, 32, 8, 128, L.NKV_KV_BF16) == size(50) > full
    # tiles that fill the chip, short contexts, prompts of many tiles, nothing known
    assert plan(16, 32768, 2048, 9000, 32, 8, 128, L.NKV_KV_BF16) == 0
    assert plan(3, 120, 40, 300, 32, 8, 128, L.NKV_KV_BF16) == 0
    assert plan(1, 20000, 20000, 30000, 32, 8, 128, L.NKV_KV_BF16) == 0
    assert plan(1, 512, 512, 0, 32, 8, 128, L.NKV_KV_BF16) == 0
    assert plan(0, 0, 0, 0, 32, 8, 128, L.NKV_KV_BF16) == 0
    assert plan(1, 512, 512, 12800, 30, 8, 128, L.NKV_KV_BF16) == 0
    # steps that the plain launch was measured faster for: tiles of head_dim 256, and rows that
    # several column groups stream; and those where the split one was still
    bf16 = L.NKV_KV_BF16
    assert plan(16, 1923, 560, 853, 16, 16, 256, bf16) == 0  # plain 55 us, split 73
    assert plan(5, 3668, 1824, 6770, 16, 16, 256, bf16) == 0  # 476, 606
    assert plan(80, 81, 2, 2132, 128, 2, 256, bf16) == 0  # 81, 129
    assert plan(150, 217, 68, 2462, 96, 1, 128, bf16) == 0  # 96, 112
    assert plan(150, 158, 9, 4398, 128, 2, 128, bf16) == 0  # 122, 182
    assert plan(40, 995, 597, 6000, 28, 4, 256, bf16) > 0  # within 20%
    for args in SPLIT_FASTER:
        assert plan(*args) > 0, args
    # positions in 32 bits: 200 rows of a million keys, not 2000 of eight
    assert plan(200, 711, 512, 1 << 20, 32, 8, 128, L.NKV_KV_BF16) == size(200)
    assert plan(2000, 2511, 512, 1 << 23, 32, 8, 128, L.NKV_KV_BF16) == 0

    def call(kv_type=L.NKV_KV_BF16, ws=1 << 12, nbytes=full, bt=1 << 12, scale=1.0):
        return lib.nkv_prefill_varlen_split(
            kv_type, 1 << 12, 32 * 128, 1 << 12, 1 << 12, 8 * 128, 8 * 128, 1 << 12, 1 << 12, bt,
            4, 4, 1, 16, 32, 8, 128, 256, 4 * 256, 1.0, scale, scale, 1 << 12, 32 * 128, ws, nbytes,
            None)
    assert call(kv_type=3) == -1
    assert call(ws=None) == -3 and call(ws=(1 << 12) + 8) == -3 and call(nbytes=full - 1) == -3
    assert call(kv_type=L.NKV_KV_FP8, bt=None) == -1  # fp8 rows are paged
    # scales belong to fp8 rows: others get to the workspace's check whatever they are
    assert call(scale=0.0, ws=None) == -3
    assert call(kv_type=L.NKV_KV_FP8, scale=0.0, ws=None) == -1
