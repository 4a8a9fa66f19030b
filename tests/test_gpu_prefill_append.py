"""Prompt attention over keys in flight with the K/V append in its launch, against the two calls: the same bits in the cache and in the
output, for token counts around what a wavefront copies, rows of one to eight heads, calls of one launch, of two (an odd group of
heads), in halves and in parts, tokens without a slot, strided rows, and forms that the general call takes."""
import pytest
import torch

pytestmark = pytest.mark.gpu
D = 128


@pytest.mark.parametrize("HQ,HKV", [(28, 4), (7, 1), (5, 1), (2, 2), (16, 8), (3, 1)])
@pytest.mark.parametrize("lens,dtype,page", [([1], torch.bfloat16, 16), ([3, 1], torch.float16, 16), ([5], torch.bfloat16, 32), ([31, 2, 300], torch.bfloat16, 16),
                                             ([1500], torch.bfloat16, 16), ([700, 64, 65], torch.float16, 48)])
def test_append_with_a_prompt(sb, dev, HQ, HKV, lens, dtype, page):
    gen = torch.Generator().manual_seed(HQ + sum(lens))
    T = sum(lens)
    pages = -(-T // page) + 2
    q = torch.randn(T, HQ, D, generator=gen).to(dtype).to(dev)
    wide = torch.randn(T + 3, 3 * HKV, D, generator=gen).to(dtype).to(dev)   # (three more tokens than the prompts', as decoding ones)
    key, value = wide[:, :HKV], wide[:, 2 * HKV:]
    slots = torch.randperm(pages * page, generator=gen)[:T + 3].to(dev)
    slots[T // 2] = -1
    cache = torch.randn(2, pages, page, HKV, D, generator=gen).to(dtype).to(dev)
    plan = sb.ops.PrefillPlan(lens, lens, dev)
    starts = torch.tensor([0] + lens).cumsum(0).int().to(dev)
    call = lambda c, out, **kw: sb.ops.swa_prefill_attention(q, key[:T], value[:T], plan=plan, kv_start32=starts, window_left=1000, out=out, **kw)
    c0 = cache.clone()
    sb.ops.kv_append(key, value, c0[0], c0[1], slots)
    want = call(c0, torch.zeros_like(q))
    assert not torch.equal(c0, cache)
    for kw in ({}, dict(n_parts=1)):                                       # (in one native step; the general call)
        c1 = cache.clone()
        got = call(c1, torch.zeros_like(q), append=(key, value, c1, slots), **kw)
        assert torch.equal(c1, c0)
        assert torch.equal(got, call(c0, torch.zeros_like(q), **kw) if kw else want)
    c1 = cache.clone()                                                     # a list of slots that only the general call takes
    got = call(c1, torch.zeros_like(q), append=(key, value, c1, slots.view(-1, 1)))
    assert torch.equal(c1, c0) and torch.equal(got, want)
    with pytest.raises(ValueError):
        call(c1, torch.zeros_like(q), append=(key, value, c1, slots[:T]))
    with pytest.raises(ValueError):
        call(c1, torch.zeros_like(q), append=(key.float(), value.float(), c1, slots))
