"""sb_swa_decode_static (split-K partials in the library's own device array, no allocation) against
sb_swa_decode with a caller workspace: both called straight through the C ABI, outputs and
log-sum-exps bit-identical (same kernels, same summation order). Two calls in a row share the
array, the second with a smaller input, so stale partials of the first are in it."""
import ctypes as C

import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(lens, bs, Hkv, D, seed):
    g = torch.Generator().manual_seed(seed)
    need = [(n + bs - 1) // bs for n in lens]
    nb = sum(need) + 3
    perm = torch.randperm(nb, generator=g)
    kv = torch.randn(2, nb, bs, Hkv, D, generator=g).bfloat16()
    tables = torch.zeros(len(lens), max(need), dtype=torch.int32)
    p = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[p:p + n]
        p += n
    return kv, tables


def _args(N, q, kv, tables, seq_lens, out, lse, wl, n_split, flags, ws):
    Hq, D = q.shape[1], q.shape[2]
    kc, vc = kv[0], kv[1]
    return N.SwaDecodeArgs(
        q=N.ptr(q), k_cache=N.ptr(kc), v_cache=N.ptr(vc), out=N.ptr(out), lse=N.ptr(lse),
        block_table=N.ptr(tables), seq_lens=N.ptr(seq_lens),
        workspace=N.ptr(ws), workspace_bytes=0 if ws is None else ws.numel(),
        num_rows=q.shape[0], num_q_heads=Hq, num_kv_heads=kc.shape[2], head_size=D, block_size=kc.shape[1],
        window_left=wl, max_seq_len=tables.shape[1] * kc.shape[1], n_split=n_split, dtype=N.SB_BF16, phases=0,
        flags=flags, scale=D ** -0.5,
        q_stride_row=q.stride(0), q_stride_head=q.stride(1),
        out_stride_row=out.stride(0), out_stride_head=out.stride(1),
        kv_stride_block=kc.stride(0), kv_stride_row=kc.stride(1), kv_stride_head=kc.stride(2),
        block_table_stride=tables.stride(0), stream=N.stream_ptr(q.device))


@pytest.mark.parametrize("flags", [0, 2])  # fixed split, balanced split (SB_DECODE_BALANCED)
def test_static_scratch_matches_workspace_call_twice(sb, dev, flags):
    N = sb._native
    L = N.lib()
    Hq, Hkv, D, bs, wl = 28, 4, 128, 16, 300
    for lens, n_split, seed in (([700, 333, 64, 1, 512, 290, 451, 97, 640, 18, 200, 305], 4, 1),
                                ([90, 411, 33], 3, 2)):        # second call: fewer rows, fewer splits
        kv, tables = _problem(lens, bs, Hkv, D, seed)
        q = torch.randn(len(lens), Hq, D, generator=torch.Generator().manual_seed(seed + 10)).bfloat16().to(dev)
        kv, tables = kv.to(dev), tables.to(dev)
        seq_lens = torch.tensor(lens, dtype=torch.int32, device=dev)
        need = L.sb_swa_decode_workspace_bytes(len(lens), Hq, D, n_split)
        assert 0 < need <= N.SB_SWA_DECODE_STATIC_SCRATCH_BYTES
        ws = torch.zeros(need, dtype=torch.uint8, device=dev)      # a workspace starts zeroed (merge counters)
        outs = []
        for fn, w in ((L.sb_swa_decode, ws), (L.sb_swa_decode_static, None)):
            out = torch.full((len(lens), Hq, D), float("nan"), dtype=torch.bfloat16, device=dev)
            lse = torch.full((len(lens), Hq), float("nan"), dtype=torch.float32, device=dev)
            a = _args(N, q, kv, tables, seq_lens, out, lse, wl, n_split, flags, w)
            rc = fn(C.byref(a))
            assert rc == 0, N.last_error()
            torch.cuda.synchronize()
            outs.append((out, lse))
        assert torch.equal(outs[0][0].view(torch.int16), outs[1][0].view(torch.int16))
        assert torch.equal(outs[0][1].view(torch.int32), outs[1][1].view(torch.int32))
        assert not torch.isnan(outs[1][0].float()).any()


def test_static_scratch_rejects_oversized_call(sb, dev):
    N = sb._native
    L = N.lib()
    rows, Hq, Hkv, D, n_split = 600, 28, 4, 128, 8
    assert L.sb_swa_decode_workspace_bytes(rows, Hq, D, n_split) > N.SB_SWA_DECODE_STATIC_SCRATCH_BYTES
    kv, tables = _problem([40] * rows, 16, Hkv, D, 3)
    q = torch.zeros(rows, Hq, D, dtype=torch.bfloat16, device=dev)
    out = torch.zeros_like(q)
    a = _args(N, q, kv.to(dev), tables.to(dev), torch.full((rows,), 40, dtype=torch.int32, device=dev), out, None,
              -1, n_split, 0, None)
    assert L.sb_swa_decode_static(C.byref(a)) == N.SB_ERR_WORKSPACE
    assert "scratch" in N.last_error()


@pytest.mark.parametrize("length,fits", [(4097, 15), (4097, 20), (400, 1), (400, 3), (400, 64)])
def test_chosen_split_follows_the_workspace(sb, dev, length, fits):
    """n_split = 0: the library never chooses more partials than the caller's workspace holds, down to runs of eight
    chunks each (15 splits of 4097 keys, 1 of 400); below that the call is refused, as an explicit split is."""
    N = sb._native
    L = N.lib()
    kv, tables = _problem([length], 16, 4, 128, 6)
    kv, tables = kv.to(dev), tables.to(dev)
    q = torch.randn(1, 28, 128, generator=torch.Generator().manual_seed(7)).bfloat16().to(dev)
    lens = torch.tensor([length], dtype=torch.int32, device=dev)
    need = L.sb_swa_decode_workspace_bytes(1, 28, 128, fits)
    ws = torch.zeros(need, dtype=torch.uint8, device=dev) if need else None
    outs = []
    for n_split, w in ((0, ws), (1, None)):
        out = torch.full((1, 28, 128), float("nan"), dtype=torch.bfloat16, device=dev)
        assert L.sb_swa_decode(C.byref(_args(N, q, kv, tables, lens, out, None, 4200, n_split, 0, w))) == 0, N.last_error()
        outs.append(out.float())
    assert (outs[0] - outs[1]).abs().max() <= 2 ** -7 * outs[1].abs().max()     # each rounds fp32 results to bf16
    if length == 4097:
        small = torch.zeros(L.sb_swa_decode_workspace_bytes(1, 28, 128, 14), dtype=torch.uint8, device=dev)
        assert L.sb_swa_decode(C.byref(_args(N, q, kv, tables, lens, out, None, 4200, 0, 0, small))) == N.SB_ERR_WORKSPACE
