"""Block form of the GLA prompt kernels at the edges of its 32-token blocks and their 16-token halves: lengths around both, one
workgroup per head and one per group of heads, with rows behind the prompt that must not be read. Tolerances as for the other
prompt tests: fp32 states 1e-4 of the largest entry, outputs 2e-2 + half a bf16 ulp + 2^-9 of the largest (bf16 operands of
the product with the state)."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import gla as G

pytestmark = pytest.mark.gpu
D = 128


def _check(o, ref_o, S, ref_S):
    o, S = o.double().cpu().numpy(), S.double().cpu().numpy()
    assert np.isfinite(o).all() and np.isfinite(S).all()
    assert np.abs(S - ref_S).max() <= 1e-4 * np.abs(ref_S).max()
    assert (np.abs(o - ref_o) <= 2e-2 + 2.0 ** -8 * np.abs(ref_o) + 2.0 ** -9 * np.abs(ref_o).max()).all()


@pytest.mark.parametrize("H,Hk,gdtype", [(3, 3, torch.float32), (3, 3, torch.bfloat16), (8, 2, torch.float32), (14, 2, torch.float16)])
@pytest.mark.parametrize("T", [1, 2, 15, 16, 17, 31, 32, 33, 47, 49, 63, 64, 65, 96, 97])
def test_lengths_around_blocks(sb, dev, T, H, Hk, gdtype):
    """A prompt of T tokens in front of one that has no slot and holds NaN: its tokens are the next rows in memory."""
    g = torch.Generator().manual_seed(T * 31 + H)
    q = torch.randn(T + 70, H, D, generator=g).bfloat16()
    k, v = (torch.randn(T + 70, Hk, D, generator=g).bfloat16() for _ in range(2))
    gate = (F.logsigmoid(torch.randn(T + 70, Hk, D, generator=g)) / 4).to(gdtype)
    S0 = torch.randn(2, Hk, D, D, generator=g) * 0.1
    rep = H // Hk
    head_first = lambda x: x[:T].float().transpose(0, 1)[None]
    wide = lambda x: head_first(x).repeat_interleave(rep, 1).numpy()
    ref_o, ref_S = G.gla_recurrent(head_first(q).numpy(), wide(k), wide(v), wide(gate), S0[:1].repeat_interleave(rep, 1).double().numpy())
    for x in (q, k, v, gate):
        x[T:] = float("nan")
    cu = torch.tensor([0, T, T + 70], dtype=torch.int32, device=dev)
    slots = torch.tensor([0, -1], dtype=torch.int32, device=dev)
    for per_head in ((None,) if rep == 1 else (True, False)):
        state = S0.to(dev)
        o = sb.ops.gla_recurrent_packed(q.to(dev), k.to(dev), v.to(dev), gate.to(dev), state, cu, slots, per_head=per_head)
        _check(o[:T].transpose(0, 1), ref_o[0], state[0], ref_S[0, ::rep])
        assert torch.equal(state[1].cpu(), S0[1])


def test_rows_too_far_apart_for_the_block_form(sb, dev):
    """Rows 64 MiB apart: 32 of them do not fit the block form's 32-bit offsets, so the call takes the step-by-step kernel."""
    T, H, step = 3, 1, 1 << 25
    g = torch.Generator().manual_seed(0)
    q, k, v = (torch.randn(T, H, D, generator=g).bfloat16() for _ in range(3))
    gate = F.logsigmoid(torch.randn(T, H, D, generator=g)) / 16
    ref_o, ref_S = G.gla_recurrent(*(x.float().transpose(0, 1)[None].numpy() for x in (q, k, v, gate)), None)

    def apart(x):
        far = torch.empty((T - 1) * step + H * D, dtype=x.dtype, device=dev).as_strided((T, H, D), (step, D, 1))
        return far.copy_(x.to(dev))

    state = torch.zeros(1, H, D, D, device=dev)
    cu = torch.tensor([0, T], dtype=torch.int32, device=dev)
    o = sb.ops.gla_recurrent_packed(apart(q), k.to(dev), v.to(dev), gate.to(dev), state, cu)
    _check(o.transpose(0, 1), ref_o[0], state[0], ref_S[0])


@pytest.mark.parametrize("H,Hk,lens", [(14, 2, [300, 257, 64, 1] + [65] * 28),   # 64 groups: 4 segments, each adds up those before it
                                       (2, 2, [1100]),                           # 17 segments: a scan adds up
                                       (28, 28, [600, 500]),                     # 4 segments per head, added up
                                       (8, 2, [97])])                            # a single prompt in segments of one block
def test_segments_start_from_what_those_before_them_add_up_to(sb, dev, H, Hk, lens):
    """Cut calls against the uncut one: the same blocks, a state rounded once more per segment (fp32: 1e-4 of the largest entry)."""
    n, T = len(lens), sum(lens)
    g = torch.Generator().manual_seed(T)
    q = torch.randn(T, H, D, generator=g).bfloat16().relu().to(dev)
    k, v = (torch.randn(T, Hk, D, generator=g).bfloat16().relu().to(dev) for _ in range(2))
    gate = (F.logsigmoid(torch.randn(T, Hk, D, generator=g)) / 16).to(dev)
    S0 = (torch.randn(n, Hk, D, D, generator=g) * 0.1).to(dev)
    cu = torch.tensor([0] + lens).cumsum(0).int().to(dev)
    st, st1 = S0.clone(), S0.clone()
    o = sb.ops.gla_recurrent_packed(q, k, v, gate, st, cu, None, max_seq_len=max(lens))
    o1 = sb.ops.gla_recurrent_packed(q, k, v, gate, st1, cu, None, max_seq_len=max(lens), per_head=True)   # (never cut)
    assert (st - st1).abs().max() <= 1e-4 * st1.abs().max()
    d, ref = (o.float() - o1.float()).abs(), o1.float().abs()
    assert (d <= 2.0 ** -7 * ref + 2.0 ** -8 * ref.max()).all()      # each rounds the same sums, and its operands, to bf16
