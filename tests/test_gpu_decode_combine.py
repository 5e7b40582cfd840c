"""The merge of a decode row's partials by one wave and by four, at partial counts around what
a wave holds and has in flight (ranges of 4 chunks = 64 tokens; up to 129 partials), and the
store at token counts around a change of its chunks per thread, against the oracle."""
import pytest
import torch

from oracle.attention_ref import paged_decode_ref, store_kvcache_ref

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("D,kind", [(128, "bf16"), (64, "fp16"), (256, "bf16")])
@pytest.mark.parametrize("ctx", [
    [8192], [8191, 1], [64 * 33], [64 * 32 + 1, 64 * 16, 0, 64 * 17],  # one to four rows: wide
    [1, 64, 65, 64 * 16 + 1] + [400] * 70,                              # one wave each
])
def test_merge_of_many_partials(nkv, dev, ctx, D, kind):
    print(ctx[:4], D, kind, flush=True)
    g = torch.Generator().manual_seed(9)
    Hq, Hk, B = 8, 2, 256
    dt = torch.float16 if kind == "fp16" else torch.bfloat16
    need = [-(-n // B) for n in ctx]
    bt = torch.full((len(ctx), 32), -1, dtype=torch.int32)  # 512 chunks wide: ranges of 4
    ids = torch.randperm(sum(need) + 1, generator=g).to(torch.int32)
    at = 0
    for i, n in enumerate(need):
        bt[i, :n] = ids[at:at + n]
        at += n
    kv = torch.randn(2, sum(need) + 1, B, Hk, D, generator=g).to(dt)
    q = (3 * torch.randn(len(ctx), Hq, D, generator=g)).to(dt)  # peaks: weights far apart
    lens = torch.tensor(ctx, dtype=torch.int32)
    out = nkv.paged_decode(q.to(dev), kv[0].to(dev), kv[1].to(dev), lens.to(dev), bt.to(dev),
                           D ** -0.5)
    torch.cuda.synchronize()
    some = [i for i in range(len(ctx)) if i < 5 or i % 9 == 0]
    ref = paged_decode_ref(q[some].float(), kv[0], kv[1], lens[some], bt[some], D ** -0.5)
    # outputs of a few units of N(0, 1) values, rounded to 16 bits, weights too
    assert (out.float().cpu()[some] - ref).abs().max().item() <= 2e-2


@pytest.mark.parametrize("kind", ["bf16", "fp16", "fp8"])
@pytest.mark.parametrize("B,width", [(16, 4), (16, 5), (256, 2), (256, 16), (256, 17)])
@pytest.mark.parametrize("batch", [1, 2, 3, 11])
def test_small_batches_in_short_ranges(nkv, dev, batch, B, width, kind):
    """Ranges of three and four chunks: batches and table widths around the changes, and
    contexts that end at and beside a range's end."""
    g = torch.Generator().manual_seed(batch * width)
    Hq, Hk, D = 8, 2, 128
    dt = torch.float16 if kind == "fp16" else torch.bfloat16
    top = B * width
    lens = torch.tensor([min(top, n) for n in (top, 48, 33, 1, 32, 49, 0, 64, 97, 31, 2)[:batch]],
                        dtype=torch.int32)
    bt = torch.randperm(batch * width, generator=g).to(torch.int32).view(batch, width)
    kv = torch.randn(2, batch * width, B, Hk, D, generator=g)
    kv = kv.to(torch.float8_e4m3fn) if kind == "fp8" else kv.to(dt)
    q = (3 * torch.randn(batch, Hq, D, generator=g)).to(dt)
    out = nkv.paged_decode(q.to(dev), kv[0].to(dev), kv[1].to(dev), lens.to(dev), bt.to(dev),
                           D ** -0.5)
    torch.cuda.synchronize()
    ref = paged_decode_ref(q.float(), kv[0].float(), kv[1].float(), lens, bt, D ** -0.5)
    assert (out.float().cpu() - ref).abs().max().item() <= 2e-2  # as above


@pytest.mark.parametrize("Hk,D,tokens", [(8, 128, 1), (8, 128, 16383), (8, 128, 16385),
                                         (1, 64, 7), (3, 128, 43691)])
def test_store_around_its_chunks_per_thread(nkv, dev, Hk, D, tokens):
    g = torch.Generator().manual_seed(tokens)
    k, v = torch.randn(2, tokens, Hk, D, generator=g).to(torch.bfloat16)
    pool = torch.zeros(2, -(-tokens // 256) + 1, 256, Hk, D, dtype=torch.bfloat16)
    slots = torch.randperm(pool.size(1) * 256, generator=g)[:tokens].to(torch.int32)
    slots[tokens // 2] = -1
    kc, vc = pool[0].to(dev), pool[1].to(dev)
    nkv.store_kvcache(k.to(dev), v.to(dev), kc, vc, slots.to(dev))
    torch.cuda.synchronize()
    store_kvcache_ref(k, v, pool[0], pool[1], slots)
    assert torch.equal(kc.cpu(), pool[0]) and torch.equal(vc.cpu(), pool[1])
