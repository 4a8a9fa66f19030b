"""The append and the round trips of a step in one launch (sb_fp8_step): the bytes of the append's own kernel, and the round
trips as the oracle computes them on the CPU."""
import pytest
import torch

from oracle import quant as Q

pytestmark = pytest.mark.gpu
NAMES = {torch.bfloat16: "bf16", torch.float16: "f16", torch.float32: "f32"}


def _rounded(x, scale):
    return torch.from_numpy(Q.fp8_round(x.float().cpu().numpy(), scale, NAMES[x.dtype])).to(x.dtype)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("tokens,heads", [(1, 1), (3, 4), (2, 5), (67, 9), (33, 4)])
@pytest.mark.parametrize("with_append", [True, False])
def test_one_launch_equals_its_parts(sb, dev, dtype, tokens, heads, with_append):
    g = torch.Generator().manual_seed(tokens * 10 + heads)
    k, v = (torch.randn(tokens, 2 * heads, 128, generator=g).to(dtype).to(dev)[:, ::2] for _ in range(2))
    q = (torch.randn(tokens, 7, 128, generator=g) * 300).to(dtype).to(dev)
    blocks = tokens // 16 + 2
    slots = torch.randperm(blocks * 16, generator=g)[:tokens]
    slots[::5] = -1
    slots = slots.to(dev)
    caches = [torch.full((2, blocks, 16, heads, 128), 9, dtype=torch.uint8, device=dev) for _ in range(2)]
    kk, vv = k.contiguous(), v.contiguous()
    if with_append:
        sb.ops.kv_append_fp8(k, v, caches[0][0], caches[0][1], slots, 0.5, 0.25)
    for rounds in ([(q, 2.0)], [(q, 2.0), (kk, 0.5), (vv, 0.25)], [(q, 1.0), (q[:0], 1.0), (vv, 0.125)]):
        caches[1].fill_(9)
        outs = sb.ops.fp8_step((k, v, caches[1][0], caches[1][1], slots, 0.5, 0.25) if with_append else None, rounds)
        assert torch.equal(caches[0], caches[1])
        for o, (x, scale) in zip(outs, rounds):
            assert o.shape == x.shape and torch.equal(o.cpu(), _rounded(x, scale))


def test_tensors_of_several_types(sb, dev):
    x = [torch.randn(5, 16, device=dev).to(t) for t in (torch.bfloat16, torch.float32, torch.float16)]
    for o, t in zip(sb.ops.fp8_step(None, [(t, 0.5) for t in x]), x):
        assert torch.equal(o.cpu(), _rounded(t, 0.5))
