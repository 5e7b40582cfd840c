"""Attention.forward's one native call against its separate store and attention calls: the same
outputs and caches bit for bit in every form that the call takes, and the separate calls'
own answers where it does not."""
import importlib
import struct
from types import SimpleNamespace

import pytest
import torch

L = importlib.import_module("nanokv-llm_amd._lib")
attention = importlib.import_module("nanokv-llm_amd.layers.attention")
FP8 = torch.float8_e4m3fn
NO_COMPRESSION = SimpleNamespace(kv_compress_enabled=False)


def _step(dev, kind, decode, views, D=128, Hq=8, Hk=2, B=64):
    """(layer, forward arguments, context arguments) of a small step."""
    g = torch.Generator().manual_seed(3)
    dt = torch.float16 if kind == "fp16" else torch.bfloat16
    new = [1] * 5 if decode else [1, 70, 1, 33]
    keys = [5, 64, 65, 300, 1] if decode else [200, 90, 1, 900]
    need = [-(-n // B) for n in keys]
    ids = torch.randperm(sum(need) + 2, generator=g).to(torch.int32)
    bt = torch.full((len(keys), max(need) + 1), -1, dtype=torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = ids[at:at + n]
        at += n
    seq = torch.repeat_interleave(torch.arange(len(new)), torch.tensor(new))
    pos = torch.cat([torch.arange(b - a, b) for a, b in zip(new, keys)])
    slots = bt[seq, pos // B] * B + (pos % B).to(torch.int32)
    slots[-1] = -1  # a padding slot
    n = sum(new)
    qkv = torch.randn(n, Hq + 2 * Hk, D, generator=g).to(dt).to(dev)
    q, k, v = qkv[:, :Hq], qkv[:, Hq:Hq + Hk], qkv[:, Hq + Hk:]
    if not views:
        q, k, v = q.contiguous(), k.contiguous(), v.contiguous()
    kv = torch.randn(2, sum(need) + 2, B, Hk, D, generator=g)
    kv = (kv * 16).to(FP8) if kind == "fp8" else kv.to(dt)
    layer = attention.Attention(Hq, D, D ** -0.5, Hk, NO_COMPRESSION, 1)
    layer.k_cache, layer.v_cache = kv.to(dev)
    if kind == "fp8":
        layer.k_scale, layer.v_scale = 1 / 16, 1 / 8
    cs = lambda x: torch.tensor([0] + x).cumsum(0).to(torch.int32).to(dev)  # noqa: E731
    ctx = (True, None, None, 0, 0, slots.to(dev), torch.tensor(keys, dtype=torch.int32).to(dev),
           bt.to(dev)) if decode else \
        (False, cs(new), cs(keys), max(new), max(keys), slots.to(dev), None, bt.to(dev))
    return layer, (q, k, v, 0), ctx


def _run(nkv, layer, args, ctx, monkeypatch=None):
    """(out, caches) of forward on copies of the layer's caches."""
    caches = [c.clone() if c.dtype != FP8 else c.view(torch.uint8).clone().view(FP8)
              for c in (layer.k_cache, layer.v_cache)]
    kept = layer.k_cache, layer.v_cache
    layer.k_cache, layer.v_cache = caches
    nkv.set_context(*ctx)
    out = layer(*args)
    torch.cuda.synchronize()
    nkv.reset_context()
    layer.k_cache, layer.v_cache = kept
    return [out] + [c.view(torch.uint8) for c in caches]


@pytest.mark.gpu
@pytest.mark.parametrize("views", [False, True])
@pytest.mark.parametrize("decode", [True, False])
@pytest.mark.parametrize("kind,D", [("bf16", 128), ("fp16", 128), ("fp8", 128), ("bf16", 64),
                                    ("fp8", 256)])
def test_one_call_equals_the_separate_calls(nkv, dev, monkeypatch, kind, D, decode, views):
    layer, args, ctx = _step(dev, kind, decode, views, D=D)
    taken = []
    step = attention.Attention._step
    monkeypatch.setattr(attention.Attention, "_step",
                        lambda self, *a: taken.append(step(self, *a)) or taken[-1])
    one = _run(nkv, layer, args, ctx)
    assert taken[0] is not None
    monkeypatch.setattr(attention.Attention, "_step", lambda self, *a: None)
    apart = _run(nkv, layer, args, ctx)
    assert one[0].shape == apart[0].shape
    assert all(torch.equal(a, b) for a, b in zip(one, apart))


@pytest.mark.gpu
def test_other_forms_keep_the_separate_calls_answers(nkv, dev):
    """What the one call does not take raises as it did, or runs as it did."""
    layer, (q, k, v, _), ctx = _step(dev, "bf16", True, False)
    with pytest.raises(ValueError):  # value of another type
        _run(nkv, layer, (q, k, v.half(), 0), ctx)
    with pytest.raises(AssertionError):  # one slot per token
        _run(nkv, layer, (q, k, v, 0), ctx[:5] + (ctx[5][:-1],) + ctx[6:])
    with pytest.raises(ValueError):  # a host tensor
        _run(nkv, layer, (q, k.cpu(), v, 0), ctx)
    # no block table: the new rows themselves
    layer, (q, k, v, _), ctx = _step(dev, "bf16", False, False)
    cu = ctx[1]
    out = _run(nkv, layer, (q, k, v, 0), (False, cu, cu, ctx[3], ctx[3], ctx[5], None, None))[0]
    ref = nkv.varlen_prefill(q, k, v, cu, cu, ctx[3], layer.scale)
    assert torch.equal(out, ref)


@pytest.mark.gpu
def test_no_longest_key_length_takes_the_plain_launch(nkv, dev):
    layer, args, ctx = _step(dev, "bf16", False, False)
    some = _run(nkv, layer, args, ctx[:4] + (0,) + ctx[5:])
    none = _run(nkv, layer, args, ctx[:4] + (None,) + ctx[5:])
    assert all(torch.equal(a, b) for a, b in zip(some, none))


@pytest.mark.gpu
@pytest.mark.parametrize("kv_stored", [False, True])
def test_a_full_card_runs_the_plain_launch(nkv, dev, kv_stored):
    """Torch's allocator limited to what a step that splits needs without its workspace."""
    g = torch.Generator().manual_seed(4)
    lens = torch.tensor([0, 130], dtype=torch.int32), torch.tensor([0, 9000], dtype=torch.int32)
    q, k, v = (torch.randn(130, h, 128, generator=g).bfloat16().to(dev) for h in (32, 8, 8))
    layer = attention.Attention(32, 128, 128 ** -0.5, 8, NO_COMPRESSION, 1)
    layer.k_cache, layer.v_cache = torch.randn(2, 36, 256, 8, 128, generator=g).bfloat16().to(dev)
    bt = torch.arange(36, dtype=torch.int32).view(1, 36).to(dev)
    slots = torch.arange(8870, 9000, dtype=torch.int32).to(dev)
    cu_q, cu_k = (x.to(dev) for x in lens)
    assert attention.varlen_prefill_workspace(q, layer.k_cache, 1, 130, 9000).numel() > 64 << 20
    nkv.set_context(False, cu_q, cu_k, 130, 9000, slots, None, bt)
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(dev).total_memory
    torch.cuda.set_per_process_memory_fraction(
        (torch.cuda.memory_reserved(dev) + (32 << 20)) / total, dev)
    try:
        out = layer(q, k, v, 0, kv_stored=kv_stored)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0, dev)
        nkv.reset_context()
    plain = nkv.varlen_prefill(q, layer.k_cache, layer.v_cache, cu_q, cu_k, 130, 128 ** -0.5,
                               block_tables=bt)
    assert torch.equal(out, plain)


def test_the_call_checks_its_arguments_on_the_host():
    lib = L.lib()
    pack = attention._ATTENTION_ARGS.pack
    assert struct.calcsize(attention._ATTENTION_ARGS.format) == 32 * 8

    def call(kv_type=0, n_seqs=4, ws=0, decode=1, heads=8, max_q=1):
        p = 1 << 12
        return lib.nkv_attention(pack(p, 1024, p, 256, p, 256, p, p, p, 4, p, 8, 8, p, p, n_seqs,
                                      max_q, heads, 2, 128, 64, 16, kv_type, decode, p, 1024, p,
                                      ws, 0, 0.1, 1.0, 1.0))
    assert lib.nkv_attention(None) == -1
    assert call(kv_type=7) == -1
    assert call(n_seqs=-1) == -1 and call(n_seqs=1 << 33) == -1 and call(heads=0) == -1
    assert call(max_q=1 << 40, decode=0) == -1
    assert call(ws=0) == L.NKV_EWORKSPACE and call(ws=64) == L.NKV_EWORKSPACE
