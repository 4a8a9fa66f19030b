"""Long prompts of a few sequences cut into segments that run side by side: packed and batched calls whose lengths lie
at the edges of the segments, against the float64 recurrence and against the uncut call. The state is formed in fp32
either way (1e-4 relative to its largest entry, one more rounding of 2^-8 where it is stored as bf16); outputs carry the
block form's bf16 operands: 2e-2 + 2^-8 |o| (rounding of the result) + 2^-9 max|o| (operand rounding of cancelling terms)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import gla as G

pytestmark = pytest.mark.gpu
D = 128


@pytest.fixture
def cuts(sb, monkeypatch):
    """Segment counts of the calls made through ops."""
    lib, seen = sb._native.lib(), []

    class Spy:
        def __getattr__(self, name):
            fn = getattr(lib, name)
            if name != "sb_gla_prompt_segments":
                return fn

            def wrapped(a):
                seen.append(fn(a))
                return seen[-1]
            return wrapped
    spy = Spy()
    monkeypatch.setattr(sb._native, "lib", lambda: spy)
    return seen


@pytest.mark.parametrize("H,Hk,gdtype,sdtype,expect", [(4, 4, torch.float32, torch.float32, 8), (2, 2, torch.bfloat16, torch.bfloat16, 8),
                                                       (8, 2, torch.float32, torch.float32, 8), (7, 1, torch.float16, torch.bfloat16, 8)])
def test_packed_prompts_cut_into_segments(sb, dev, cuts, H, Hk, gdtype, sdtype, expect):
    n = H // Hk
    lens = [512, 449, 1, 0, 64, 65, 128, 100]        # segments of 64 tokens; slot 4 of the list is skipped
    total = sum(lens)
    g = torch.Generator().manual_seed(H)
    q = torch.randn(total, H, D, generator=g).bfloat16().relu()
    k = torch.randn(total, Hk, D, generator=g).bfloat16().relu()
    v = torch.randn(total, Hk, D, generator=g).bfloat16()
    gate = (F.logsigmoid(torch.randn(total, Hk, D, generator=g)) / 16).to(gdtype)
    state = (torch.randn(10, Hk, D, D, generator=g) * 0.02).to(sdtype)
    slots = [9, 0, 7, 3, -1, 5, 2, 1]
    cu = torch.tensor([0] + list(np.cumsum(lens)), dtype=torch.int32).to(dev)
    st = state.to(dev)
    out = torch.full((total, H, D), 7.0, dtype=torch.bfloat16, device=dev)
    dq, dk, dv, dg = (x.to(dev) for x in (q, k, v, gate))
    idx = torch.tensor(slots, dtype=torch.int32, device=dev)
    sb.ops.gla_recurrent_packed(dq, dk, dv, dg, st, cu, idx, out=out, max_seq_len=512)
    assert cuts == [expect]
    st1, out1 = state.to(dev), torch.full_like(out, 7.0)
    sb.ops.gla_recurrent_packed(dq, dk, dv, dg, st1, cu, idx, out=out1, max_seq_len=512, per_head=True)
    assert cuts == [expect, 1]
    rtol = 1e-4 if sdtype == torch.float32 else 2.0 ** -8
    assert (st.double() - st1.double()).abs().max() <= rtol * st1.double().abs().max()
    got_o, got_s = out.float().cpu().numpy(), st.double().cpu().numpy()
    for i, L in enumerate(lens):
        a = int(sum(lens[:i]))
        if slots[i] < 0:
            assert (got_o[a:a + L] == 7.0).all()
            continue
        if L == 0:
            continue
        t = lambda x: np.repeat(x[a:a + L].transpose(0, 1)[None].float().numpy(), 1, 0)
        r = lambda x: np.repeat(t(x), n, 1)
        ref_o, ref_s = G.gla_recurrent(t(q), r(k), r(v), r(gate), np.repeat(state[slots[i]][None].double().numpy(), n, 1))
        assert np.abs(got_s[slots[i]] - ref_s[0, ::n]).max() <= rtol * np.abs(ref_s).max(), i
        ref = ref_o[0].transpose(1, 0, 2)
        assert (np.abs(got_o[a:a + L] - ref) <= 2e-2 + 2.0 ** -8 * np.abs(ref) + 2.0 ** -9 * np.abs(ref).max()).all(), i
    rest = [s for s in range(10) if s not in slots] + [3]
    assert np.array_equal(got_s[rest], state.double().numpy()[rest])


@pytest.mark.parametrize("H,Hk", [(2, 2), (8, 2)])
def test_batched_prompt_cut_into_segments(sb, dev, cuts, H, Hk):
    """[B, H, T, D] views of token-major tensors, a last segment of 5 tokens, state by batch row."""
    B, T, n = 2, 517, H // Hk
    g = torch.Generator().manual_seed(T)
    q = torch.randn(B, T, H, D, generator=g).bfloat16().relu().transpose(1, 2)
    k, v = (torch.randn(B, T, Hk, D, generator=g).bfloat16().relu().transpose(1, 2) for _ in range(2))
    gate = (F.logsigmoid(torch.randn(B, T, Hk, D, generator=g)) / 16).transpose(1, 2)
    o, s = sb.fused_recurrent_gla(q.to(dev), k.to(dev), v.to(dev), gate.to(dev), output_final_state=True)
    assert cuts and cuts[0] > 1
    r = lambda x: np.repeat(x.float().numpy(), n, 1)
    ref_o, ref_s = G.gla_recurrent(q.float().numpy(), r(k), r(v), r(gate), None)
    assert np.abs(s.double().cpu().numpy() - ref_s[:, ::n]).max() <= 1e-4 * np.abs(ref_s).max()
    got = o.float().cpu().numpy()
    assert (np.abs(got - ref_o) <= 2e-2 + 2.0 ** -8 * np.abs(ref_o) + 2.0 ** -9 * np.abs(ref_o).max()).all()


@pytest.mark.parametrize("H,Hk", [(2, 2), (8, 2)])
def test_prompt_longer_than_the_stated_bound(sb, dev, cuts, H, Hk):
    """The bound only sizes the cut: the last segment takes what is left, and nothing outside the workspace is touched."""
    lens = [900, 40]
    g = torch.Generator().manual_seed(1)
    q = torch.randn(sum(lens), H, D, generator=g).bfloat16().relu().to(dev)
    k, v = (torch.randn(sum(lens), Hk, D, generator=g).bfloat16().relu().to(dev) for _ in range(2))
    gate = (F.logsigmoid(torch.randn(sum(lens), Hk, D, generator=g)) / 16).to(dev)
    state = (torch.randn(2, Hk, D, D, generator=g) * 0.02).to(dev)
    cu = torch.tensor([0, 900, 940], dtype=torch.int32, device=dev)
    st, st1 = state.clone(), state.clone()
    o = sb.ops.gla_recurrent_packed(q, k, v, gate, st, cu, None, max_seq_len=512)
    o1 = sb.ops.gla_recurrent_packed(q, k, v, gate, st1, cu, None, max_seq_len=900, per_head=True)
    assert cuts[0] > 1 and cuts[1] == 1
    assert (st - st1).abs().max() <= 1e-4 * st1.abs().max()
    d, ref = (o.float() - o1.float()).abs(), o1.float().abs()
    assert (d <= 2.0 ** -7 * ref + 2.0 ** -8 * ref.max()).all()      # each rounds the same sums, and its operands, to bf16


@pytest.mark.parametrize("lens,bound,cut", [([100] * 8, None, False), ([100] * 8, 100, False), ([800], None, True), ([800] * 2, None, True),
                                            ([800] * 2, 800, True), ([1000, 100, 100], None, True), ([10, 0, 0, 0, 0, 2000], None, True)])
def test_prompts_of_unstated_length(sb, dev, cuts, lens, bound, cut):
    """Without max_seq_len only the total of all prompts is known: many short prompts must not be cut as one long one
    (every segment but the first would be empty, behind two more launches)."""
    B, T = len(lens), sum(lens)
    g = torch.Generator().manual_seed(B)
    q = torch.randn(T, 28, D, generator=g).bfloat16().relu().to(dev)
    k, v = (torch.randn(T, 4, D, generator=g).bfloat16().relu().to(dev) for _ in range(2))
    gate = (F.logsigmoid(torch.randn(T, 4, D, generator=g)) / 16).to(dev)
    state = torch.zeros(B, 4, D, D, device=dev)
    cu = torch.tensor([0] + lens).cumsum(0).int().to(dev)
    o = sb.gla_prefill_packed(q, k, v, gate, state, torch.arange(B, device=dev), cu, B, max_query_len=bound)
    assert any(n > 1 for n in cuts) == cut
    state1 = torch.zeros_like(state)
    o1 = sb.ops.gla_recurrent_packed(q, k, v, gate, state1, cu, per_head=True)      # (never cut)
    assert (state - state1).abs().max() <= 1e-4 * state1.abs().max()
    d, ref = (o.float() - o1.float()).abs(), o1.float().abs()
    assert (d <= 2.0 ** -7 * ref + 2.0 ** -8 * ref.max()).all()
