"""Decode over a byte-code cache with the append in the launch, against the append (and the queries' fp8 round trip) in front of it:
the same codes, scales and outputs to the bit, at every place a newest key can have in a chunk, for rows whose last chunk is in the
first, a middle or the only split, for rows without a slot, without keys, and with rows of zeros, of the largest values and of
infinities."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D, PAGE = 14, 2, 128, 16
LENS = [1, 2, 15, 16, 17, 31, 32, 33, 47, 48, 49, 64, 65, 300, 1025, 0, 40, 90]
NO_SLOT = (16, 17)                                                         # the last two rows store nothing


@pytest.mark.parametrize("kv", ["int8", "fp8"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("window,n_split", [(-1, 0), (-1, 1), (-1, 7), (40, 3), (0, 1)])
def test_append_codes(sb, dev, kv, dtype, window, n_split):
    gen = torch.Generator().manual_seed(LENS[3] + n_split)
    R, width = len(LENS), -(-max(LENS) // PAGE)
    table = torch.randperm(R * width, generator=gen).view(R, width).int().to(dev)
    lens = torch.tensor(LENS, dtype=torch.int32, device=dev)
    last = (lens - 1).clamp(min=0)
    slots = table[torch.arange(R, device=dev), (last // PAGE).long()].long() * PAGE + (last % PAGE)
    slots[list(NO_SLOT)] = -1
    q = torch.randn(R, HQ, D, generator=gen).to(dtype).to(dev)
    key, value = (torch.randn(R, 3 * HKV, D, generator=gen).to(dtype).to(dev)[:, HKV:2 * HKV] for _ in range(2))
    key[3], value[4], key[5], value[6] = 0, 0, torch.finfo(dtype).max, torch.finfo(dtype).max / 4
    key[15, 0, 7] = float("inf")                                           # (a row without keys of its own: stored, not attended to)
    shape = (2, R * width, PAGE, HKV, D)
    codes = torch.randint(-127, 128, shape, dtype=torch.int8, generator=gen).to(dev)
    scales = (torch.rand(2, R * width, HKV, PAGE, generator=gen) * 0.02).to(dev)
    if kv == "fp8":
        codes = torch.randn(shape, generator=gen).to(torch.float8_e4m3fn).to(dev)
    q_scale = 0.37 if kv == "fp8" else 0.0
    extra = lambda s: dict(k_scale=s[0], v_scale=s[1]) if kv == "int8" else dict(fp8_scales=(0.5, 2.0))
    call = lambda q, c, s, **kw: sb.ops.swa_decode_attention(q, c[0], c[1], lens, block_table=table, window_left=window, n_split=n_split,
                                                             balanced=False, return_lse=True, **extra(s), **kw)
    c0, s0 = codes.clone(), scales.clone()
    rounded = q
    if kv == "int8":
        sb.ops.kv_append_int8(key, value, c0[0], c0[1], s0[0], s0[1], slots)
    else:
        sb.ops.kv_append_fp8(key, value, c0[0], c0[1], slots, 0.5, 2.0)
        rounded = sb.ops.fp8_round(q, q_scale)
    want, want_lse = call(rounded, c0, s0)
    c1, s1 = codes.clone(), scales.clone()
    got, lse = call(q, c1, s1, new_key=key, new_value=value, new_slot_mapping=slots, append_codes=q_scale)
    assert torch.equal(c1.view(torch.uint8), c0.view(torch.uint8)) and torch.equal(s1, s0)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16)) and torch.equal(lse.view(torch.int32), want_lse.view(torch.int32))
    assert torch.isfinite(got[7:]).all() and not torch.equal(c1.view(torch.uint8), codes.view(torch.uint8))


@pytest.mark.parametrize("kv", ["int8", "fp8"])
@pytest.mark.parametrize("softcap,alibi", [(20.0, False), (0.0, True), (20.0, True)])
def test_append_codes_with_score_options(sb, dev, kv, softcap, alibi):
    """The same with a soft cap, slopes or both on the scores (of the calls with the append in front, test_gpu_score_options has the values)."""
    gen = torch.Generator().manual_seed(7)
    R, width = len(LENS), -(-max(LENS) // PAGE)
    table = torch.randperm(R * width, generator=gen).view(R, width).int().to(dev)
    lens = torch.tensor(LENS, dtype=torch.int32, device=dev)
    last = (lens - 1).clamp(min=0)
    slots = table[torch.arange(R, device=dev), (last // PAGE).long()].long() * PAGE + (last % PAGE)
    q, key, value = (torch.randn(R, h, D, generator=gen).bfloat16().to(dev) for h in (HQ, HKV, HKV))
    shape = (2, R * width, PAGE, HKV, D)
    codes, scales = torch.randint(-127, 128, shape, dtype=torch.int8, generator=gen).to(dev), torch.full((2, R * width, HKV, PAGE), 0.02, device=dev)
    if kv == "fp8":
        codes = torch.randn(shape, generator=gen).to(torch.float8_e4m3fn).to(dev)
    slopes = torch.linspace(0.01, 0.3, HQ, device=dev) if alibi else None
    how = dict(k_scale=scales[0], v_scale=scales[1]) if kv == "int8" else dict(fp8_scales=(0.5, 2.0))
    call = lambda c, **kw: sb.ops.swa_decode_attention(q, c[0], c[1], lens, block_table=table, window_left=200, balanced=False, return_lse=True,
                                                       softcap=softcap, alibi_slopes=slopes, **how, **kw)
    c0, s0 = codes.clone(), scales.clone()
    got, lse = call(codes, new_key=key, new_value=value, new_slot_mapping=slots, append_codes=0.0)
    if kv == "int8":
        sb.ops.kv_append_int8(key, value, c0[0], c0[1], s0[0], s0[1], slots)
        assert torch.equal(scales, s0)
        how = dict(k_scale=s0[0], v_scale=s0[1])
    else:
        sb.ops.kv_append_fp8(key, value, c0[0], c0[1], slots, 0.5, 2.0)
    want, want_lse = call(c0)
    assert torch.equal(codes.view(torch.uint8), c0.view(torch.uint8))
    assert torch.equal(got, want) and torch.equal(lse.view(torch.int32), want_lse.view(torch.int32))
    plain = sb.ops.swa_decode_attention(q, c0[0], c0[1], lens, block_table=table, window_left=200, balanced=False, **how)
    assert torch.isfinite(got).all() and not torch.equal(plain, want)


@pytest.mark.parametrize("kv", ["int8", "fp8"])
def test_layer_call_under_capture(sb, dev, kv):
    """A decode layer over byte codes through the backend: eager (native step and general form) and replayed from a graph."""
    R, keys, width = 3, 3000, 188
    meta = lambda: sb.MetaAttentionMetadata(
        num_prefills=0, num_prefill_tokens=0, num_decode_tokens=R, slot_mapping=slots, seq_lens=None, seq_lens_tensor=lens,
        max_prefill_seq_len=0, max_decode_seq_len=keys, context_lens_tensor=None, block_tables=table, use_cuda_graph=True,
        max_query_len=1, max_decode_query_len=1)
    gen = torch.Generator().manual_seed(5)
    table = torch.randperm(R * width, generator=gen).view(R, width).int().to(dev)
    lens = torch.tensor([3000, 17, 1600], dtype=torch.int32, device=dev)
    slots = table[torch.arange(R, device=dev), ((lens - 1) // PAGE).long()].long() * PAGE + (lens - 1) % PAGE
    q, k, v = (torch.randn(R, h, D, generator=gen).bfloat16().to(dev) for h in (HQ, HKV, HKV))
    if kv == "int8":
        cache = sb.Int8KVCache.allocate(R * width, PAGE, HKV, D, dev)
        cache.codes.random_(-127, 128)
        cache.scales.uniform_(0.0, 0.02)
        copy = lambda: sb.Int8KVCache(cache.codes.clone(), cache.scales.clone())
        held = lambda c: (c.codes, c.scales)
    else:
        cache = torch.randn(2, R * width, PAGE, HKV, D, generator=gen).to(torch.float8_e4m3fn).to(dev)
        copy, held = cache.clone, lambda c: (c.view(torch.uint8),)
    impl = sb.MetaAttentionImpl(HQ, D, D ** -0.5, HKV, None, 2048, "fp8" if kv == "fp8" else "auto")
    layer = type("Layer", (), dict(_q_scale_float=0.5) if kv == "fp8" else {})()
    run = lambda q, c, out: impl.forward(layer, q, k, v, None, None, None, c, meta(), out)
    spread = torch.randn(R, 2 * HQ, D, device=dev).bfloat16()
    spread[:, :HQ] = q
    for _ in range(2):                                                     # (the first allocates the scratch memory)
        c0, c1, c2 = copy(), copy(), copy()
        want = run(q, c0, torch.zeros_like(q)).clone()
        general = run(spread[:, :HQ], c1, torch.zeros_like(q))             # fp8: the unfused form
        assert torch.equal(general, want) and all(torch.equal(a, b) for a, b in zip(held(c1), held(c0)))
    if kv == "fp8":                                                        # (0 would mean no round trip)
        layer._q_scale_float = 0.0
        with pytest.raises(ValueError):
            run(q, c1, torch.zeros_like(q))
        layer._q_scale_float = 0.5
    out = torch.zeros_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(q, c2, out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        run(q, c1, torch.zeros_like(q))
        torch.cuda.synchronize()
        assert torch.equal(out, want) and all(torch.equal(a, b) for a, b in zip(held(c2), held(c0)))
    sb.ops.release_graph_workspace()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("T,rounded,heads", [(1, 1, 1), (9, 4, 4), (70, 70, 5), (33, 31, 2)])
def test_append_that_rounds(sb, dev, dtype, T, rounded, heads):
    """The rows of a prompt as the INT8 cache holds them, from the append's own launch: the bits of append and round trips by themselves."""
    gen = torch.Generator().manual_seed(T)
    key, value = (torch.randn(T, 3 * heads, D, generator=gen).to(dtype).to(dev)[:, heads:2 * heads] for _ in range(2))
    key[0, 0] = 0
    value[T - 1] *= 1e4
    slots = torch.randperm(96, generator=gen)[:T].to(dev)
    slots[T // 2] = -1
    codes, scales = torch.zeros(2, 6, PAGE, heads, D, dtype=torch.int8, device=dev), torch.zeros(2, 6, heads, PAGE, device=dev)
    c1, s1 = codes.clone(), scales.clone()
    sb.ops.kv_append_int8(key, value, codes[0], codes[1], scales[0], scales[1], slots)
    k, v = sb.ops.kv_append_int8(key, value, c1[0], c1[1], s1[0], s1[1], slots, rounded)
    assert torch.equal(c1, codes) and torch.equal(s1, scales) and k.shape == (rounded, heads, D)
    assert torch.equal(k, sb.ops.quantize_sym(key[:rounded])) and torch.equal(v, sb.ops.quantize_sym(value[:rounded]))
    with pytest.raises(ValueError):
        sb.ops.kv_append_int8(key, value, c1[0], c1[1], s1[0], s1[1], slots, T + 1)
