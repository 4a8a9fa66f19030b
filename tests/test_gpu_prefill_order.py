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
