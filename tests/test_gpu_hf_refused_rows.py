"""A Hugging Face decode call whose new keys or values the cache refuses, or whose copy fails, leaves the cache as it was: the next call
gives the bits of a cache that never saw it. Where only the attention fails the rows are in the cache, as after an update by itself."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D, W = 4, 2, 128, 32
# rows a full window takes behind it before they are moved to the front of their memory; 80 without a window fill it, so that the next has new memory
ROOM = {W: 64, None: 80}


def _rows(dev, B, n, seed, heads=HKV, dtype=torch.bfloat16, dim=D):
    return torch.randn(B, n, heads, dim, generator=torch.Generator().manual_seed(seed)).to(dtype).to(dev).transpose(1, 2)


def _bad(dev, B, how):
    good, shape = _rows(dev, B, 1, 90), {}
    if how == "type":
        shape = dict(dtype=torch.float16)
    elif how == "heads":
        shape = dict(heads=HKV + 1)
    elif how == "size":
        shape = dict(dim=64)
    if how == "device":
        return good, good.cpu()
    if how == "batch":
        return _rows(dev, B + 1, 1, 91), _rows(dev, B + 1, 1, 92)
    return (good, _rows(dev, B, 1, 91, **shape)) if how != "heads" else (_rows(dev, B, 1, 91, **shape),) * 2


@pytest.mark.parametrize("how", ["type", "heads", "size", "device", "batch", "memory"])
@pytest.mark.parametrize("B", [1, 3])
@pytest.mark.parametrize("window,steps", [(W, 3), (W, ROOM[W]), (None, ROOM[None])])
def test_refused_rows_leave_the_cache_as_it_was(sb, dev, monkeypatch, how, B, window, steps):
    """`steps` valid tokens, then one that is refused: into memory with room behind the rows, at a move to the front of it, and at a
    move to new memory. `memory`: an allocation of the copy fails (a batch of rows out of one wider tensor is laid out anew)."""
    kw = {} if window else dict(cache_window_size=None)
    caches = [sb.Cache(), sb.Cache()]
    first = _rows(dev, B, window or 16, 1), _rows(dev, B, window or 16, 2)
    for c in caches:
        c.update(attn_state=first, layer_idx=0, offset=first[0].shape[2], cache_kwargs={"window_size": window})
    call = lambda c, q, k, v: sb.sliding_window_attention(q, k, v, W, c, 0, **kw)
    q = _rows(dev, B, 1, 3, heads=HQ)
    for i in range(steps):
        for c in caches:
            call(c, q, _rows(dev, B, 1, 100 + i), _rows(dev, B, 1, 300 + i))
    before = [x.clone() for x in caches[0][0]["attn_state"]]
    if how == "memory":
        def out_of_memory(*a):
            raise torch.OutOfMemoryError("no memory for the copy")
        with monkeypatch.context() as m:
            m.setattr(sb.ops, "window_shift_pair", out_of_memory)
            m.setattr(sb.ops, "dense_decode", lambda *a: None)
            with pytest.raises(torch.OutOfMemoryError):
                call(caches[0], q, _rows(dev, B, 1, 90), _rows(dev, B, 1, 91))
    else:
        with pytest.raises((ValueError, RuntimeError)):
            call(caches[0], q, *_bad(dev, B, how))
    assert all(torch.equal(x, y) for x, y in zip(caches[0][0]["attn_state"], before))
    for i in range(2):
        got, want = (call(c, q, _rows(dev, B, 1, 500 + i), _rows(dev, B, 1, 600 + i)) for c in caches)
        assert torch.equal(got, want)
        assert all(torch.equal(x, y) for x, y in zip(caches[0][0]["attn_state"], caches[1][0]["attn_state"]))


def test_rows_are_kept_where_the_attention_fails(sb, dev):
    cache, other = sb.Cache(), sb.Cache()
    first = _rows(dev, 2, W, 1), _rows(dev, 2, W, 2)
    q, k, v = _rows(dev, 2, 1, 3, heads=HQ), _rows(dev, 2, 1, 4), _rows(dev, 2, 1, 5)
    for c in (cache, other):
        c.update(attn_state=first, layer_idx=0, offset=W, cache_kwargs={"window_size": W})
    other.update(attn_state=(k, v), layer_idx=0, offset=1, cache_kwargs={"window_size": W})
    with pytest.raises((ValueError, RuntimeError)):
        sb.sliding_window_attention(q.half(), k, v, W, cache, 0)
    with pytest.raises((ValueError, RuntimeError)):                        # a mask without a row per sequence
        sb.sliding_window_attention(q, k, v, W, other, 0, torch.ones(1, W, dtype=torch.long, device=dev))
    cache.update(attn_state=(k, v), layer_idx=0, offset=1, cache_kwargs={"window_size": W})
    assert all(torch.equal(x, y) for x, y in zip(cache[0]["attn_state"], other[0]["attn_state"]))


def test_a_replaced_update_is_called(sb, dev, monkeypatch):
    """An `update` put in place of the cache's own, on the object or on the class, sees every decode call."""
    cache, seen, original = sb.Cache(), [], sb.Cache.update
    first = _rows(dev, 1, W, 1), _rows(dev, 1, W, 2)
    cache.update(attn_state=first, layer_idx=0, offset=W, cache_kwargs={"window_size": W})
    q, k, v = _rows(dev, 1, 1, 3, heads=HQ), _rows(dev, 1, 1, 4), _rows(dev, 1, 1, 5)
    cache.update = lambda *a, **kw: seen.append("object") or original(cache, *a, **kw)
    sb.sliding_window_attention(q, k, v, W, cache, 0)
    del cache.update
    monkeypatch.setattr(sb.Cache, "update", lambda self, *a, **kw: seen.append("class") or original(self, *a, **kw))
    sb.sliding_window_attention(q, k, v, W, cache, 0)
    assert seen == ["object", "class"]
