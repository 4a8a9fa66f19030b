"""Lengths and bounds of a dense left-padded batch in one launch (sb_dense_rows), and the K/V shift as one launch
(sb_window_shift_pair), against the same arithmetic in torch on the CPU: whole numbers and bytes, compared exactly."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cols", [1, 63, 64, 1023, 1025, 3072, 3073, 4096, 4097, 9001])
@pytest.mark.parametrize("dtype", [torch.int64, torch.int32, torch.int16, torch.bool, torch.uint8, torch.float32, torch.bfloat16])
def test_dense_rows(sb, dev, cols, dtype):
    gen = torch.Generator().manual_seed(cols)
    B, Q, extra = 3, 1 + cols % 5, cols % 3
    K = cols + extra                       # a mask shorter than the keys counts the missing entries as padding
    mask = torch.ones(B + 1, cols + 7)     # a spare row, and a slice with a row stride of its own
    for b in range(B):
        mask[b, :7 + int(torch.randint(0, cols + 1, (1,), generator=gen))] = 0
    mask = mask.to(dtype)
    if dtype.is_floating_point:
        mask[0, :8] = -0.0
    pad = (K - (mask[:B, -cols:] != 0).sum(dim=1)).to(torch.int32)
    sliced = mask.to(dev)[:, -cols:]
    for m in (sliced, sliced.t().contiguous().t()):
        seq_lens, row_seq, key_lo, kv_start = sb.ops.dense_rows(B, Q, K, 1000, dev, m)
        assert torch.equal(seq_lens.cpu(), (K - Q + 1 + torch.arange(Q)).int().repeat(B))
        assert torch.equal(row_seq.cpu(), torch.arange(B).int().repeat_interleave(Q))
        assert torch.equal(key_lo.cpu(), pad.repeat_interleave(Q))
        assert torch.equal(kv_start.cpu(), torch.arange(B) * 1000)


def test_dense_rows_without_mask_and_many_queries(sb, dev):
    seq_lens, row_seq, key_lo, kv_start = sb.ops.dense_rows(2, 2500, 3000, 0, dev)
    assert key_lo is None and torch.equal(kv_start.cpu(), torch.zeros(2, dtype=torch.int64))
    assert torch.equal(seq_lens.cpu(), (501 + torch.arange(2500)).int().repeat(2))
    assert torch.equal(row_seq.cpu(), torch.arange(2).int().repeat_interleave(2500))
    with pytest.raises(ValueError):
        sb.ops.dense_rows(2, 1, 4, 0, dev, torch.ones(1, 4, device=dev))


def test_mask_without_columns_hides_every_key(sb, dev):
    """An empty tensor has no address, which is not the same as no mask."""
    empty = torch.ones(2, 0, dtype=torch.int64, device=dev)
    assert sb.ops.dense_rows(2, 3, 4, 0, dev, empty)[2].tolist() == [4] * 6
    q, k = torch.randn(2, 4, 1, 64, device=dev), torch.randn(2, 2, 1, 64, device=dev)
    assert bool((sb.sliding_window_attention(q, k, k, 8, attention_mask=empty) == 0).all())


@pytest.mark.parametrize("v_keep", [5, 3])   # the same rows in both (one launch), and not (two)
def test_window_shift_pair(sb, dev, v_keep):
    gen = torch.Generator().manual_seed(0)
    old = torch.randn(2, 2, 3, 20, 64, generator=gen)
    new = torch.randn(2, 2, 3, 4, 64, generator=gen)
    src, fresh, dst = old.to(dev), new.to(dev), torch.zeros(2, 2, 3, 24, 64, device=dev)
    sb.ops.window_shift_pair((src[0], dst[0], fresh[0], 5, 7, 2), (src[1], dst[1], fresh[1], v_keep, 7, 2))
    want = torch.zeros(2, 2, 3, 24, 64)
    for i, keep in enumerate((5, v_keep)):
        want[i, :, :, 2:2 + keep] = old[i, :, :, 7:7 + keep]
        want[i, :, :, 2 + keep:6 + keep] = new[i]
    assert torch.equal(dst.cpu(), want)


def test_refused_append_leaves_the_cache_as_it_was(sb, dev):
    cache = sb.Cache()
    k = torch.randn(1, 2, 6, 64, device=dev)
    cache.update(attn_state=(k, k), layer_idx=0, offset=6, cache_kwargs={"window_size": 8})
    bad = torch.randn(1, 2, 1, 64, device=dev, dtype=torch.bfloat16)
    with pytest.raises(ValueError):
        cache.update(attn_state=(k[:, :, :1], bad), layer_idx=0, offset=1, cache_kwargs={"window_size": 8})
    kk, vv = cache.update(attn_state=(k[:, :, :1], k[:, :, 1:2]), layer_idx=0, offset=1, cache_kwargs={"window_size": 8})["attn_state"]
    assert torch.equal(kk, torch.cat([k, k[:, :, :1]], 2)) and torch.equal(vv, torch.cat([k, k[:, :, 1:2]], 2))
