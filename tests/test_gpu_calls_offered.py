"""Calls in a form that the native layer steps do not have (other head sizes, more than 16 query heads per kv head, fp32 decode,
score options, float masks, large batches) go to the general form at once: an attempt costs them 1 to 4 us for nothing."""
import pytest
import torch

pytestmark = pytest.mark.gpu
PAGE = 16


def _layer(sb, dev, HQ=8, HKV=2, D=128, dtype=torch.bfloat16, alibi=None, cap=None):
    table, lens = torch.arange(4, dtype=torch.int32, device=dev).view(2, 2), torch.tensor([20, 9], dtype=torch.int32, device=dev)
    q, k, v = (torch.randn(2, h, D, device=dev).to(dtype) for h in (HQ, HKV, HKV))
    cache = torch.randn(2, 4, PAGE, HKV, D, device=dev).to(dtype)
    slots = torch.tensor([19, 40], device=dev)
    meta = sb.MetaAttentionMetadata(
        num_prefills=0, num_prefill_tokens=0, num_decode_tokens=2, slot_mapping=slots, seq_lens=None, seq_lens_tensor=lens, max_prefill_seq_len=0,
        max_decode_seq_len=20, context_lens_tensor=None, block_tables=table, use_cuda_graph=True, max_query_len=1, max_decode_query_len=1)
    impl = sb.MetaAttentionImpl(HQ, D, D ** -0.5, HKV, alibi, 2048, "auto", logits_soft_cap=cap)
    out, ref = torch.empty_like(q), torch.empty_like(q)
    impl.forward(type("Layer", (), {})(), q, k, v, None, None, None, cache, meta, out)
    if alibi is None and cap is None:                                      # (the cache holds the new rows by now)
        sb.ops.swa_decode_attention(q, cache[0], cache[1], lens, block_table=table, window_left=2047, out=ref, balanced=False)
        assert torch.allclose(out.float(), ref.float(), rtol=1e-2, atol=1e-2)   # (fp32, other sizes: the same kernel; 16 bit: one rounding)


def _hugging_face(sb, dev, B=2, D=128, dtype=torch.bfloat16, mask=None):
    cache = sb.Cache()
    rows = torch.randn(B, 2, 8, D, device=dev).to(dtype)
    cache.update(attn_state=(rows, rows), layer_idx=0, offset=8, cache_kwargs={"window_size": 8})
    q, k, v = (torch.randn(B, h, 1, D, device=dev).to(dtype) for h in (4, 2, 2))
    out = sb.sliding_window_attention(q, k, v, 8, cache, 0, mask)
    assert out.shape == (B, 1, 4, D) and torch.isfinite(out).all()


@pytest.mark.parametrize("form", ["head size", "heads", "fp32", "alibi", "cap", "hf head size", "hf batch", "hf mask"])
def test_forms_that_are_not_offered(sb, dev, monkeypatch, form):
    offered, real = [], sb._native.calls()

    class Watch:
        def __getattr__(self, name):
            return lambda *a: offered.append(name) or getattr(real, name)(*a)

    monkeypatch.setattr(sb._native, "calls", lambda: Watch())
    if form == "head size":
        _layer(sb, dev, D=64)
    elif form == "heads":
        _layer(sb, dev, HQ=20, HKV=1)
    elif form == "fp32":
        _layer(sb, dev, dtype=torch.float32)
    elif form == "alibi":
        _layer(sb, dev, alibi=[0.1] * 8)
    elif form == "cap":
        _layer(sb, dev, cap=20.0)
    elif form == "hf head size":
        _hugging_face(sb, dev, D=64)
    elif form == "hf batch":
        _hugging_face(sb, dev, B=65)
    else:
        _hugging_face(sb, dev, mask=torch.ones(2, 8, device=dev))
    assert not {"decode", "dense_decode"} & set(offered)
