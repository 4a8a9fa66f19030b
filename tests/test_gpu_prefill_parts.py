"""Prompt attention with the keys of a tile cut into parts (fp32 partials and a merge) and with workgroups of two heads:
against float64 attention, over dense keys and over paged element and byte-code caches, in bf16 and fp16. Outputs are rounded
from fp32 and the probabilities on the way: 1e-2 (bf16) or 1.25e-3 (fp16, three more bits) of the 2-norm, the same bound for cut
and uncut calls and between the two. Their log-sum-exps come from the same fp32 scores, summed in another order: terms of up to
1100 keys, each within 2^-24 of itself, move the logarithm by 6.6e-5 at most, and a value below 16 has places of 1e-6: 1e-4."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128
BOUND = {torch.bfloat16: 1e-2, torch.float16: 1.25e-3}


def _reference(q, k, v, lens, ctx, window, key_lo, G):
    outs, at, kat = [], 0, 0
    for s, n in enumerate(lens):
        L = n + ctx
        qq, kk, vv = q[at:at + n].double(), k[kat:kat + L].double().repeat_interleave(G, 1), v[kat:kat + L].double().repeat_interleave(G, 1)
        sc = torch.matmul(qq.transpose(0, 1), kk.permute(1, 2, 0).contiguous()) * D ** -0.5
        pos, key = torch.arange(n)[:, None] + ctx, torch.arange(L)[None]
        hide = (key > pos) | (key < key_lo[s])
        if window >= 0:
            hide |= key < pos - window
        sc.masked_fill_(hide, float("-inf"))
        p = torch.nan_to_num(torch.softmax(sc, -1))
        outs.append(torch.matmul(p, vv.transpose(0, 1).contiguous()).transpose(0, 1))
        at, kat = at + n, kat + L
    return torch.cat(outs)


@pytest.mark.parametrize("G", [1, 2, 3, 4, 5, 7, 8])
@pytest.mark.parametrize("lens,ctx,window", [([1], 0, -1), ([65], 300, -1), ([64, 3], 257, 100), ([130, 1, 70], 0, 4096), ([40], 1000, 511)])
@pytest.mark.parametrize("n_parts,dtype", [(n, torch.bfloat16) for n in (0, 1, 2, 3, 7, 40)] + [(3, torch.float16)])
def test_parts_and_pairs(sb, dev, G, lens, ctx, window, n_parts, dtype):
    g = torch.Generator().manual_seed(G * 100 + n_parts)
    Hkv, T, Lk = 2, sum(lens), sum(lens) + ctx * len(lens)
    q, k, v = (torch.randn(n, h, D, generator=g).to(dtype) for n, h in ((T, Hkv * G), (Lk, Hkv), (Lk, Hkv)))
    key_lo = [(7 * s) % (n + ctx + 2) for s, n in enumerate(lens)]      # some rows see nothing: zeros
    kv_start = torch.tensor([0] + [n + ctx for n in lens]).cumsum(0)[:-1].to(dev)
    run = lambda parts: sb.ops.swa_prefill_attention(
        q.to(dev), k.to(dev), v.to(dev), query_lens=lens, seq_lens_k=[n + ctx for n in lens], kv_start=kv_start,
        key_lo=torch.tensor(key_lo, dtype=torch.int32, device=dev), window_left=window, return_lse=True, n_parts=parts)
    out, lse = run(n_parts)
    ref = _reference(q, k, v, lens, ctx, window, key_lo, G)
    assert (out.cpu().double() - ref).norm() <= BOUND[dtype] * ref.norm()
    if n_parts == 1:
        return
    out1, lse1 = run(1)
    assert (out.double() - out1.double()).norm() <= BOUND[dtype] * out1.double().norm()
    assert torch.equal(torch.isneginf(lse), torch.isneginf(lse1))
    ok = ~torch.isneginf(lse)
    assert (lse[ok] - lse1[ok]).abs().max() <= 1e-4


def test_starts_as_32_bit_values(sb, dev):
    g = torch.Generator().manual_seed(2)
    lens = [70, 5, 130]
    q, k, v = (torch.randn(sum(lens), h, D, generator=g).bfloat16().to(dev) for h in (4, 2, 2))
    starts = torch.tensor([0] + lens).cumsum(0)
    run = lambda **kw: sb.ops.swa_prefill_attention(q, k, v, query_lens=lens, window_left=64, **kw)
    a = run(kv_start=starts[:-1].contiguous().to(dev))
    assert torch.equal(a, run(kv_start32=starts.int().to(dev))) and torch.equal(a, run())
    for bad in (starts.to(dev), starts[:2].int().to(dev)):
        with pytest.raises(ValueError):
            run(kv_start32=bad)


@pytest.mark.parametrize("kv", ["bf16", "int8", "fp8"])
def test_paged_parts_with_meta_rows_and_options(sb, dev, kv):
    """The parts over a paged cache (element and byte codes), with meta rows (walked by the first part) and score options,
    against float64 attention over the dequantised rows (the soft cap's exp2 and reciprocal are of the hardware's precision,
    2^-22 of a score of at most 20: 5e-6 more)."""
    g = torch.Generator().manual_seed(5)
    Hkv, G, bs, n, ctx = 2, 4, 16, 50, 500
    L = n + ctx
    blocks = (L + bs - 1) // bs
    table = torch.randperm(blocks, generator=g).int()[None].to(dev)
    q = torch.randn(n, Hkv * G, D, generator=g).bfloat16().to(dev)
    kw = {}
    if kv == "int8":
        cache = torch.randint(-127, 128, (2, blocks, bs, Hkv, D), generator=g).to(torch.int8).to(dev)
        sc = (torch.rand(2, blocks, Hkv, bs, generator=g) * 0.02 + 0.005).to(dev)
        kw.update(k_scale=sc[0], v_scale=sc[1])
    elif kv == "fp8":
        cache = torch.randn(2, blocks, bs, Hkv, D, generator=g).to(torch.float8_e4m3fn).to(dev)
        kw.update(fp8_scales=(0.5, 2.0))
    else:
        cache = torch.randn(2, blocks, bs, Hkv, D, generator=g).bfloat16().to(dev)
    meta = torch.randn(2, 37, Hkv, D, generator=g).bfloat16().to(dev)
    kw.update(meta_k=meta[0], meta_v=meta[1], softcap=20.0, alibi_slopes=torch.linspace(0.01, 0.3, Hkv * G, device=dev))
    run = lambda parts: sb.ops.swa_prefill_attention(q, cache[0], cache[1], query_lens=[n], seq_lens_k=[L], block_table=table,
                                                     window_left=400, return_lse=True, n_parts=parts, **kw)
    order = table[0].long().cpu()
    rows = cache.cpu().float()[:, order].flatten(1, 2)[:, :L]                       # as the kernel takes them: rounded to bf16
    if kv == "int8":
        rows = (rows * sc.cpu()[:, order].permute(0, 1, 3, 2).flatten(1, 2)[:, :L, :, None]).bfloat16()
    elif kv == "fp8":
        rows = (rows * torch.tensor([0.5, 2.0])[:, None, None, None]).bfloat16()
    keys, values = (torch.cat([m.cpu().double(), r.double()]).repeat_interleave(G, 1) for m, r in zip(meta, rows))
    score = torch.einsum("nhd,khd->hnk", q.cpu().double(), keys) * D ** -0.5
    slope = torch.linspace(0.01, 0.3, Hkv * G).double()[:, None, None]
    pos, key, m = torch.arange(n)[:, None], torch.arange(L)[None], torch.arange(37)[None]
    dist = torch.cat([(pos + 37 - n - m).abs(), pos + ctx - key], 1)                # meta rows: one stacked sequence of n queries
    score = 20 * torch.tanh(score / 20) - slope * dist
    score.masked_fill_(torch.cat([torch.zeros(n, 37, dtype=torch.bool), (key > pos + ctx) | (key < pos + ctx - 400)], 1), float("-inf"))
    ref, ref_lse = torch.einsum("hnk,khd->nhd", torch.softmax(score, -1), values), torch.logsumexp(score, -1).t()
    one, lse1 = run(1)
    for parts in (1, 2, 5):
        out, lse = run(parts)
        assert (out.cpu().double() - ref).norm() <= BOUND[torch.bfloat16] * ref.norm()
        assert (lse.cpu().double() - ref_lse).abs().max() <= 1e-4
        assert (out.float() - one.float()).norm() <= 5e-3 * one.float().norm()   # both round the same sums to bf16
        assert (lse - lse1).abs().max() <= 1e-4


def test_parted_call_under_capture(sb, dev):
    g = torch.Generator().manual_seed(9)
    q = torch.randn(100, 28, D, generator=g).bfloat16().to(dev)
    k, v = torch.randn(2100, 4, D, generator=g).bfloat16().to(dev), torch.randn(2100, 4, D, generator=g).bfloat16().to(dev)
    plan, start = sb.ops.PrefillPlan([100], [2100], dev), torch.zeros(1, dtype=torch.int64, device=dev)
    out = torch.empty_like(q)
    run = lambda: sb.ops.swa_prefill_attention(q, k, v, plan=plan, kv_start=start, window_left=4096, out=out)
    run()
    eager = out.clone()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run()
    for _ in range(3):
        out.zero_()
        torch.randn(1 << 20, device=dev).sum()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(out, eager)


@pytest.mark.parametrize("parts", [2, 3, 5, 8])
def test_infinite_value_in_the_last_part(sb, dev, parts):
    """An infinite value that all queries see makes the output infinite, cut or not: the merge fills the rest of a trip
    to memory with the last part again, which must not count (infinity times 0 is a NaN)."""
    g = torch.Generator().manual_seed(parts)
    n, ctx = 40, 600
    q, k, v = (torch.randn(m, h, D, generator=g).bfloat16() for m, h in ((n, 4), (n + ctx, 2), (n + ctx, 2)))
    v[ctx - 5, :, 7] = float("inf")
    kw = dict(query_lens=[n], seq_lens_k=[n + ctx], kv_start=torch.zeros(1, dtype=torch.int64, device=dev), window_left=-1)
    whole, cut = (sb.ops.swa_prefill_attention(q.to(dev), k.to(dev), v.to(dev), n_parts=m, **kw).float().cpu() for m in (1, parts))
    assert torch.isposinf(whole[:, :, 7]).all() and torch.isposinf(cut[:, :, 7]).all()
    assert torch.equal(torch.isfinite(whole), torch.isfinite(cut))


def test_more_parts_than_the_merge_addresses(sb, dev):
    """Eight rows of a head's partials are addressed with 32 bits: 511 parts at 1024 heads. A call that asks for more gets fewer,
    and from as many parts as the walk has chunks on the cut is the same: the same bits."""
    g = torch.Generator().manual_seed(4)
    q, k, v = (torch.randn(n, h, D, generator=g).bfloat16().to(dev) for n, h in ((1, 1024), (300, 64), (300, 64)))
    run = lambda n: sb.ops.swa_prefill_attention(q, k, v, query_lens=[1], seq_lens_k=[300], kv_start=torch.zeros(1, dtype=torch.int64, device=dev),
                                                 window_left=4096, n_parts=n)
    assert torch.equal(run(1024), run(40))


@pytest.mark.parametrize("kv", ["dense", "paged", "int8", "fp8"])
@pytest.mark.parametrize("G,lens,ctx,window", [(7, [257], 0, 4096), (7, [1300], 0, 4096), (3, [65, 300], 520, 300), (2, [64], 256, 4096), (1, [290, 31], 64, -1),
                                               (5, [33], 700, 290)])
def test_halves_of_a_walk(sb, dev, kv, G, lens, ctx, window):
    """Workgroups whose two sets of wavefronts each take half of the keys: odd and even numbers of chunks, a last group of one head,
    walks whose second half is all masked for some tokens, more workgroups than CUs (1300 tokens), and the same call cut into two
    parts, each against float64 attention element by element. A probability is rounded to bf16 (2^-8 of itself, its sum is not), so an
    output lies within 2^-8 of the same average over |v|, and 2^-8 of itself from its own rounding; scores of up to 128 terms in
    fp32 move both by less than 2^-12. The log-sum-exps come from the same fp32 scores (as above)."""
    g = torch.Generator().manual_seed(G + len(lens))
    Hkv, T, keys = 4, sum(lens), [n + ctx for n in lens]
    q = torch.randn(T, Hkv * G, D, generator=g).bfloat16().to(dev)
    kw = dict(query_lens=lens, seq_lens_k=keys, window_left=window, return_lse=True)
    if kv == "dense":
        k, v = (torch.randn(sum(keys), Hkv, D, generator=g).bfloat16().to(dev) for _ in range(2))
        kw.update(kv_start=torch.tensor([0] + keys).cumsum(0)[:-1].to(dev), key_lo=torch.tensor([5] * len(lens), dtype=torch.int32, device=dev))
    else:
        width = max(-(-n // 16) for n in keys)
        table = torch.randperm(len(lens) * width, generator=g).view(len(lens), width).int()
        shape = (2, table.numel(), 16, Hkv, D)
        if kv == "paged":
            k, v = torch.randn(shape, generator=g).bfloat16().to(dev)
        elif kv == "int8":
            k, v = torch.randint(-127, 128, shape, generator=g).to(torch.int8).to(dev)
            s = (torch.rand(2, table.numel(), Hkv, 16, generator=g) * 0.02).to(dev)
            kw.update(k_scale=s[0], v_scale=s[1])
        else:
            k, v = torch.randn(shape, generator=g).to(torch.float8_e4m3fn).to(dev)
            kw.update(fp8_scales=(1.0, 1.0))
        kw.update(block_table=table.to(dev))
    plan = sb.ops.PrefillPlan(lens, keys, "cpu")
    args = sb._native.SwaPrefillArgs(num_tiles=plan.num_tiles, num_q_heads=Hkv * G, num_kv_heads=Hkv, window_left=window, tile_keys=plan.tile_keys_ptr)
    assert sb._native.lib().sb_swa_prefill_halves(ctypes.byref(args), plan.max_k, 1) == 1
    (whole, lse), (cut, lse1) = (sb.ops.swa_prefill_attention(q, k, v, n_parts=n, **kw) for n in (1, 2))
    rows = [x.cpu() for x in (k, v)]
    if kv != "dense":                                                       # as the kernel takes them: in sequence, rounded to bf16
        rows = [x.float() * (s[i].cpu().permute(0, 2, 1)[..., None] if kv == "int8" else 1.0) for i, x in enumerate(rows)]
        rows = [torch.cat([x[t.long()].flatten(0, 1)[:n] for t, n in zip(table, keys)]).bfloat16() for x in rows]
    ref = _reference(q.cpu(), rows[0], torch.cat([rows[1], rows[1].abs()], -1), lens, ctx, window, [5 if kv == "dense" else 0] * len(lens), G)
    ref, bound = ref[..., :D], (2 ** -8 + 2 ** -12) * (ref[..., D:] + ref[..., :D].abs())
    for out in (whole, cut):
        assert ((out.cpu().double() - ref).abs() <= bound).all()
    ok = ~torch.isneginf(lse1)
    assert torch.equal(torch.isneginf(lse), ~ok) and (lse[ok] - lse1[ok]).abs().max() <= 1e-4
