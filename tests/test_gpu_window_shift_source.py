"""window_shift moves rows between two buffers of one type and shape, and refuses a source that is another's: counted in the
destination's elements its rows would lie elsewhere, in part behind its end."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,shape,row0,keep", [(torch.bfloat16, (2, 2, 8, 64), 0, 4), (torch.float16, (2, 2, 8, 64), 0, 4), (torch.float32, (2, 1, 8, 64), 0, 4),
                                                   (torch.float32, (2, 2, 8, 32), 0, 4), (torch.float32, (2, 2, 8, 64), 5, 4), (torch.float32, (2, 2, 8, 64), -1, 4),
                                                   (torch.float32, (2, 2, 8, 64), 2, -1)])
def test_other_sources_are_refused(sb, dev, dtype, shape, row0, keep):
    dst = torch.zeros(2, 2, 16, 64, device=dev)
    with pytest.raises(ValueError):
        sb.ops.window_shift(torch.ones(shape, dtype=dtype, device=dev), dst, torch.ones(2, 2, 1, 64, device=dev), keep_rows=keep, src_row0=row0, dst_row0=0)
    assert not dst.any()


@pytest.mark.parametrize("old,new", [(torch.bfloat16, torch.float16), (torch.bfloat16, torch.float32), (torch.float32, torch.bfloat16)])
def test_a_full_buffer_refuses_rows_of_another_type(sb, dev, old, new):
    cache = sb.Cache()
    rows = lambda n, t: torch.randn(2, 2, n, 64, generator=torch.Generator().manual_seed(n)).to(t).to(dev)
    first = rows(8, old), rows(8, old)
    cache.update(attn_state=first, layer_idx=0, offset=8, cache_kwargs={})
    room = cache.dense_layout(0)[2] - 8
    cache.update(attn_state=(rows(room, old),) * 2, layer_idx=0, offset=room, cache_kwargs={})
    before = [x.clone() for x in cache[0]["attn_state"]]
    with pytest.raises(ValueError):
        cache.update(attn_state=(rows(1, new),) * 2, layer_idx=0, offset=1, cache_kwargs={})
    assert all(x.dtype == old and torch.equal(x, y) for x, y in zip(cache[0]["attn_state"], before))
    cache.update(attn_state=(rows(1, old),) * 2, layer_idx=0, offset=1, cache_kwargs={})
    assert torch.equal(cache[0]["attn_state"][0], torch.cat([before[0], rows(1, old)], 2))
