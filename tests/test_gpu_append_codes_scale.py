"""A query scale that is positive as the Python number it comes as, but 0 in the 32 bits the kernels take, is refused by the
decode call with its fp8 append as it is by the round trip itself: 0 there means that queries are not rounded."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D, PAGE = 4, 2, 128, 16


@pytest.mark.parametrize("scale", [1e-46, 5e-324])
@pytest.mark.parametrize("native", [True, False])
def test_scale_that_is_zero_in_32_bits(sb, dev, monkeypatch, scale, native):
    table, lens = torch.arange(2, dtype=torch.int32, device=dev).view(1, 2), torch.tensor([20], dtype=torch.int32, device=dev)
    q, k, v = (torch.randn(1, h, D, device=dev).bfloat16() for h in (HQ, HKV, HKV))
    cache = torch.randn(2, 2, PAGE, HKV, D, device=dev).to(torch.float8_e4m3fn)
    before = cache.clone()
    if not native:
        monkeypatch.setattr(sb._native, "calls", lambda: type("Off", (), dict(__getattr__=lambda self, name: lambda *a: None))())
    with pytest.raises(ValueError):
        sb.ops.fp8_step(None, [(q, scale)])
    meta = sb.MetaAttentionMetadata(
        num_prefills=0, num_prefill_tokens=0, num_decode_tokens=1, slot_mapping=torch.tensor([19], device=dev), seq_lens=None, seq_lens_tensor=lens,
        max_prefill_seq_len=0, max_decode_seq_len=20, context_lens_tensor=None, block_tables=table, use_cuda_graph=True, max_query_len=1,
        max_decode_query_len=1)
    impl = sb.MetaAttentionImpl(HQ, D, D ** -0.5, HKV, None, 2048, "fp8")
    layer = type("Layer", (), dict(_q_scale_float=scale))()
    with pytest.raises(ValueError):
        impl.forward(layer, q, k, v, None, None, None, cache, meta, torch.empty_like(q))
    with pytest.raises(ValueError):
        sb.ops.swa_decode_attention(q, cache[0], cache[1], lens, block_table=table, fp8_scales=(1.0, 1.0), out=torch.empty_like(q), balanced=False,
                                    new_key=k, new_value=v, new_slot_mapping=torch.tensor([19], device=dev), append_codes=scale)
    torch.cuda.synchronize()
    assert torch.equal(cache.view(torch.uint8), before.view(torch.uint8))
