"""The layer calls that go from tensors to the library in one native step, against the general forms of the same calls (the native
step switched off): the same kernels with the same arguments, so the same bits, over the types, strides and options it accepts; and
what it does not accept is left to the general form, which takes it or raises as it always has."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D = 14, 2, 128


@pytest.fixture
def both(sb, monkeypatch):
    """run(fn): fn's result with the native step and without it, and whether the step took the calls it was offered."""
    real, taken = sb._native.calls(), []

    class Watch:
        def __getattr__(self, name):
            def wrapped(*a):
                taken.append((name, getattr(real, name)(*a)))
                return taken[-1][1]
            return wrapped

    class Off:
        def __getattr__(self, name):
            return lambda *a: None

    def run(fn, expect=True):
        taken.clear()
        monkeypatch.setattr(sb._native, "calls", lambda: Watch())
        a = fn()
        assert taken and all((r is not None) == expect for _, r in taken), [(n, type(r)) for n, r in taken]
        monkeypatch.setattr(sb._native, "calls", lambda: Off())
        b = fn()
        monkeypatch.setattr(sb._native, "calls", lambda: real)
        for x, y in zip(a, b):
            assert x.shape == y.shape and x.stride() == y.stride() and x.dtype == y.dtype and torch.equal(x, y)
    return run


def _rand(dev, *shape, dtype=torch.bfloat16, seed=0):
    return torch.randn(*shape, generator=torch.Generator().manual_seed(seed + len(shape) + shape[0])).to(dtype).to(dev)


def _pages(dev, R, keys, kv):
    width = -(-keys // 16)
    table = torch.randperm(R * width, generator=torch.Generator().manual_seed(R)).view(R, width).int().to(dev)
    shape = (2, R * width, 16, HKV, D)
    if kv == "int8":
        return table, torch.randint(-127, 128, shape, dtype=torch.int8, device=dev), torch.rand(2, R * width, HKV, 16, device=dev) * 0.02
    if kv == "fp8":
        return table, _rand(dev, *shape).to(torch.float8_e4m3fn), None
    return table, _rand(dev, *shape, dtype=torch.bfloat16 if kv == "bf16" else torch.float16), None


@pytest.mark.parametrize("kv", ["bf16", "fp16", "int8", "fp8"])
@pytest.mark.parametrize("R,keys", [(1, 40), (3, 2000), (70, 300)])
def test_paged_decode(sb, dev, both, kv, R, keys):
    table, cache, scales = _pages(dev, R, keys, kv)
    lens = torch.randint(1, keys + 1, (R,), device=dev, dtype=torch.int32)
    q = _rand(dev, R, 2 * HQ, D, dtype=torch.float16 if kv == "fp16" else torch.bfloat16)[:, :HQ]      # (rows of a wider tensor)
    extra = dict(k_scale=scales[0], v_scale=scales[1]) if kv == "int8" else dict(fp8_scales=(0.5, 2.0)) if kv == "fp8" else {}
    general = lambda **kw: (sb.ops.swa_decode_attention(q, cache[0], cache[1], lens, block_table=table, window_left=511,
                                                        out=torch.zeros(R, HQ, D, device=dev, dtype=q.dtype), **extra, **kw),)
    general(balanced=False)                                                # (the stream's scratch memory is there from here on)
    both(lambda: general(balanced=False))
    both(lambda: general(balanced=False, max_seq_len=keys, scale=0.3))
    if kv in ("bf16", "fp16"):
        general(balanced=True)
        both(lambda: general(balanced=True))
        new = [_rand(dev, R, HKV, D, dtype=q.dtype, seed=s) for s in (1, 2)]
        slots = (table[torch.arange(R, device=dev), (lens - 1) // 16].long() * 16 + (lens - 1) % 16).contiguous()

        def append():
            c = cache.clone()
            o = sb.ops.swa_decode_attention(q, c[0], c[1], lens, block_table=table, window_left=-1, out=torch.zeros(R, HQ, D, device=dev, dtype=q.dtype),
                                            new_key=new[0], new_value=new[1], new_slot_mapping=slots, balanced=False)
            return o, c
        append()
        both(append)


@pytest.mark.parametrize("kv", ["bf16", "int8", "fp8"])
def test_appends(sb, dev, both, kv):
    table, cache, scales = _pages(dev, 2, 100, kv)
    key, value = (_rand(dev, 9, 3 * HKV, D, seed=s)[:, HKV:2 * HKV] for s in (1, 2))
    slots = torch.tensor([3, -1, 5, 100, 17, 18, 19, 20, 40], device=dev)

    def run():
        c, s = cache.clone(), None if scales is None else scales.clone()
        if kv == "bf16":
            sb.ops.kv_append(key, value, c[0], c[1], slots)
        elif kv == "int8":
            sb.ops.kv_append_int8(key, value, c[0], c[1], s[0], s[1], slots)
        else:
            return sb.ops.fp8_step((key, value, c[0], c[1], slots, 0.5, 2.0), [(_rand(dev, 9, HQ, D), 0.25)])[0], c.view(torch.uint8)
        return (c,) if s is None else (c, s)
    both(run)


@pytest.mark.parametrize("paged", [False, True])
@pytest.mark.parametrize("lens,ctx", [([5], 0), ([300, 64, 1], 0), ([70], 900)])
def test_prompts(sb, dev, both, paged, lens, ctx):
    keys = [n + ctx for n in lens]
    plan = sb.ops.PrefillPlan(lens, keys, dev)
    q = _rand(dev, sum(lens), HQ, D)
    kw = dict(window_left=4096)
    if paged:
        table, cache, _ = _pages(dev, len(lens), max(keys), "bf16")
        k, v = cache[0], cache[1]
        kw.update(block_table=table)
    else:
        k, v = (_rand(dev, sum(keys), HKV, D, seed=s) for s in (1, 2))
        starts = torch.tensor([0] + keys, device=dev).cumsum(0)[:-1].contiguous()
        kw.update(**({"kv_start": starts} if ctx else {"kv_start32": starts.int()}))
    both(lambda: (sb.ops.swa_prefill_attention(q, k, v, plan=plan, out=torch.zeros_like(q), **kw),))


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("mask,B,W", [(None, 3, 256), (torch.long, 3, 256), (torch.bool, 1, 40), (torch.int32, 64, 33), (torch.int16, 5, 1)])
def test_hugging_face_decode(sb, dev, both, dtype, mask, B, W):
    rows = [_rand(dev, B, HKV, W + 3, D, dtype=dtype, seed=s) for s in (1, 2)]
    m = None
    if mask is not None:
        m = torch.ones(B, W + 9, dtype=mask, device=dev)
        m[B // 2, :9 + W // 3] = 0
    new = [_rand(dev, B, 1, h, D, dtype=dtype, seed=h).transpose(1, 2) for h in (HQ, HKV, HKV)]

    def run():
        cache = sb.Cache()
        cache.update(attn_state=tuple(rows), layer_idx=0, offset=W + 3, cache_kwargs={"window_size": W})
        outs = [sb.sliding_window_attention(*new, W, cache, 0, m) for _ in range(2)]
        return outs + list(cache[0]["attn_state"])
    run()                                                                  # (the stream's scratch memory is there from here on)
    both(run)


@pytest.mark.parametrize("B,H,n", [(1, 1, 5), (1, 3, 5), (2, 1, 5), (3, 2, 1), (2, 4, 70)])
@pytest.mark.parametrize("layout", ["transposed", "fused", "contiguous"])
def test_new_rows(sb, dev, both, B, H, n, layout):
    """A prompt's rows into a window buffer, also where they have to be laid out first."""
    wide = _rand(dev, B, n, 3 * H, D, seed=n)
    k, v = (wide[:, :, i * H:(i + 1) * H] for i in (1, 2)) if layout == "fused" else (wide[:, :, i * H:(i + 1) * H].contiguous() for i in (1, 2))
    k, v = (x.transpose(1, 2).contiguous() if layout == "contiguous" else x.transpose(1, 2) for x in (k, v))

    def push():
        storage = [torch.zeros(B, H, n + 9, D, dtype=k.dtype, device=dev) for _ in range(2)]
        sb.ops.window_shift_pair((None, storage[0], k, 0, 0, 4), (None, storage[1], v, 0, 0, 4))
        assert torch.equal(storage[0][:, :, 4:4 + n], k) and torch.equal(storage[1][:, :, 4:4 + n], v)
        assert not storage[0][:, :, :4].any() and not storage[1][:, :, 4 + n:].any()
        return storage
    both(push)


@pytest.mark.parametrize("H,Hk,sdtype", [(4, 4, torch.float32), (14, 2, torch.bfloat16)])
@pytest.mark.parametrize("slots", [None, [2, -1, 0]])
def test_linear_attention(sb, dev, both, H, Hk, sdtype, slots):
    S0 = (_rand(dev, 4, Hk, D, D, dtype=torch.float32) * 0.1).to(sdtype)
    idx = None if slots is None else torch.tensor(slots, dtype=torch.int32, device=dev)
    q = _rand(dev, 3, 1, 2 * H, D).transpose(1, 2)[:, :H]
    k, v = (_rand(dev, 3, Hk, 1, D, seed=s) for s in (1, 2))
    g = -torch.rand(3, Hk, 1, D, device=dev)

    def step():
        st = S0.clone()
        return sb.my_fused_recurrent_gla(q, k, v, g, st, idx), st
    both(step)
    lens = [300, 1, 33]
    pq, pk, pv = _rand(dev, 334, H, D), _rand(dev, 334, Hk, D, seed=1), _rand(dev, 334, Hk, D, seed=2)
    pg = -torch.rand(334, Hk, D, device=dev) / 4
    cu = torch.tensor([0] + lens).cumsum(0).int().to(dev)

    def prompts():
        st = S0.clone()
        o = sb.ops.gla_recurrent_packed(pq, pk, pv, pg, st, cu, idx, max_seq_len=300)
        if slots is not None:
            o[300:301] = 0                                                 # (rows of a prompt without a slot are left as allocated)
        return o, st
    both(prompts)


def test_other_forms_are_left_to_the_general_calls(sb, dev, both):
    table, cache, _ = _pages(dev, 3, 64, "bf16")
    lens = torch.full((3,), 50, dtype=torch.int32, device=dev)
    q, out = _rand(dev, 3, HQ, D), torch.zeros(3, HQ, D, device=dev, dtype=torch.bfloat16)
    call = lambda **kw: sb.ops.swa_decode_attention(**{**dict(q=q, key_cache=cache[0], value_cache=cache[1], seq_lens=lens, block_table=table,
                                                              window_left=-1, out=out, balanced=False), **kw})
    with pytest.raises(ValueError):
        call(q=_rand(dev, 3, HQ, D, dtype=torch.float16))
    with pytest.raises(ValueError):
        call(seq_lens=lens.long())
    with pytest.raises(ValueError):
        call(out=out[:2])
    with pytest.raises(ValueError):
        call(block_table=table.long())
    with pytest.raises(ValueError):
        call(new_key=_rand(dev, 4, HKV, D), new_value=_rand(dev, 4, HKV, D), new_slot_mapping=torch.arange(3, device=dev))
    for kw in (dict(new_value=q[:, :HKV]), dict(new_slot_mapping=torch.arange(3, device=dev)), dict(new_key=q[:, :HKV])):
        with pytest.raises(ValueError):
            call(**kw)                                                     # (the three go together)
    with pytest.raises(ValueError):
        call(q=_rand(dev, 3, 13, D), out=out[:, :13])                      # 13 query heads over 2 kv heads
    with pytest.raises(RuntimeError):
        call(q=q.cpu())
    with pytest.raises(ValueError):
        sb.ops.kv_append(q, q, cache[0], cache[1], torch.zeros(3, dtype=torch.long, device=dev))
    with pytest.raises(ValueError):
        sb.my_fused_recurrent_gla(*(_rand(dev, 2, 2, 1, D) for _ in range(3)), -torch.rand(2, 2, 1, D, device=dev),
                                  torch.zeros(1, 2, D, D, device=dev), None)  # one slot for two rows
    # accepted by the general form only: a last dimension that is not contiguous is refused by both, a slot list of two dimensions is not
    slots = torch.arange(3, device=dev).view(3, 1)
    key = _rand(dev, 3, HKV, D)
    both(lambda: (lambda c: sb.ops.kv_append(key, key, c[0], c[1], slots) or (c,))(cache.clone()), expect=False)


def test_native_step_under_capture(sb, dev):
    """A captured call keeps its scratch memory with its graph: the general form takes it."""
    table, cache, _ = _pages(dev, 2, 3000, "bf16")
    lens = torch.tensor([3000, 1700], dtype=torch.int32, device=dev)
    q = _rand(dev, 2, HQ, D)
    run = lambda out: sb.ops.swa_decode_attention(q, cache[0], cache[1], lens, block_table=table, window_left=-1, out=out, balanced=False)
    want, out = run(torch.zeros_like(q)).clone(), torch.zeros_like(q)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        run(out)
    for _ in range(3):
        out.zero_()
        graph.replay()
        run(torch.zeros_like(q))
        torch.cuda.synchronize()
        assert torch.equal(out, want)
    sb.ops.release_graph_workspace()
