"""The order in which the prefill kernel's workgroups take tiles, kv heads and head groups must not matter: a list of
1024 tiles or more (kept in sequence order, dealt in buckets of four) against the same sequences in two calls of shorter
lists (dealt latest tile first), bit for bit, for group sizes of one launch (7 = 4 + 3, 11 = 4 + 4 + 3) and of two
(6 = 4 + 2), with tile counts that leave partial eighths and buckets."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("G,Hkv", [(7, 1), (11, 2), (6, 1)])
@pytest.mark.parametrize("extra", [0, 64 * 5 + 1])
def test_long_list_equals_short_lists(sb, dev, G, Hkv, extra):
    D, wl = 128, 90
    lens = [40000, 333, 64, 1, 25500 + extra]
    cut = 1                                    # first call: one sequence of 625 tiles; second: the rest
    T = sum(lens)
    assert sum(-(-n // 64) for n in lens) >= 1024 > 625
    g = torch.Generator(device=dev).manual_seed(extra + G)
    q = torch.randn(T, G * Hkv, D, device=dev, generator=g).bfloat16()
    k, v = (torch.randn(T, Hkv, D, device=dev, generator=g).bfloat16() for _ in range(2))
    whole = sb.ops.swa_prefill_attention(q, k, v, query_lens=lens, window_left=wl)
    at = sum(lens[:cut])
    for a, b, part in ((0, at, lens[:cut]), (at, T, lens[cut:])):
        got = sb.ops.swa_prefill_attention(q[a:b], k[a:b], v[a:b], query_lens=part, window_left=wl)
        assert torch.equal(got, whole[a:b])


@pytest.mark.parametrize("HQ,Hkv", [(6, 6), (8, 4), (6, 2), (7, 1)])
@pytest.mark.parametrize("lens,ctx,window", [([1500], 700, 300), ([700, 64, 333], 900, 4096), ([2100], 0, 4096), ([65, 1, 700] * 4, 40, 4096)])
def test_short_lists_in_either_order(sb, dev, HQ, Hkv, lens, ctx, window):
    """Which of a plan's two lists a call takes, and in what order its workgroups take the heads, goes by the walks and
    the group size; the bits do not: against the same call with the dealt list alone, and with lists of the caller's own."""
    g = torch.Generator(device=dev).manual_seed(HQ)
    keys = [n + ctx for n in lens]
    q = torch.randn(sum(lens), HQ, 128, device=dev, generator=g).bfloat16()
    k, v = (torch.randn(sum(keys), Hkv, 128, device=dev, generator=g).bfloat16() for _ in range(2))
    start = torch.tensor([0] + keys, device=dev).cumsum(0)[:-1].contiguous()
    plan, dealt, own = (sb.ops.PrefillPlan(lens, keys, dev) for _ in range(3))
    dealt.tile_seq = dealt.tile_seq.clone()   # (no longer the plan's own: the call knows neither its keys nor the other list)
    turn = torch.randperm(own.num_tiles, generator=torch.Generator().manual_seed(1)).to(dev)
    own.tile_seq, own.tile_q0 = own.tile_seq[turn].contiguous(), own.tile_q0[turn].contiguous()
    a, b, c = (sb.ops.swa_prefill_attention(q, k, v, plan=p, kv_start=start, window_left=window, n_parts=1) for p in (plan, dealt, own))
    assert torch.equal(a, b) and torch.equal(a, c)
