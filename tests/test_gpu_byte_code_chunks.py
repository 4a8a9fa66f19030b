"""The byte-code decode kernel at the edges of its chunk loop: runs of 1 to 6 chunks, windows that start and end anywhere in
a chunk, block sizes that are no power of two, stale scales behind the window. Against float64 attention over the
dequantised rows; bf16 rounds the probabilities and the outputs: 2^-7 of the largest value."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D = 14, 2, 128


@pytest.mark.parametrize("kv", ["int8", "fp8"])
@pytest.mark.parametrize("block", [16, 48, 80])
@pytest.mark.parametrize("n_split", [1, 2, 3])
def test_chunk_edges(sb, dev, kv, block, n_split):
    g = torch.Generator().manual_seed(block + n_split)
    lens = [1, 15, 16, 17, 31, 32, 33, 63, 64, 65, 95, 97, 128, 129, 160, 161, 192, 200, 333]
    window = 170
    need = [(n + block - 1) // block for n in lens]
    table = torch.zeros(len(lens), max(need), dtype=torch.int32)
    perm, at = torch.randperm(sum(need), generator=g).int(), 0
    for b, n in enumerate(need):
        table[b, :n] = perm[at:at + n]
        at += n
    q = torch.randn(len(lens), HQ, D, generator=g).bfloat16()
    kw = {}
    if kv == "int8":
        codes = torch.randint(-127, 128, (2, sum(need), block, HKV, D), generator=g).to(torch.int8)
        scales = torch.rand(2, sum(need), HKV, block, generator=g) * 0.02 + 0.005
        rows = codes.double() * scales.permute(0, 1, 3, 2)[..., None].double()
        for b, n in enumerate(lens):       # stale scales of rows that hold no key yet must not reach the result
            if n % block:
                scales[:, table[b, need[b] - 1], :, n % block:] = float("nan")
        kw = dict(k_scale=scales[0].to(dev), v_scale=scales[1].to(dev))
    else:
        codes = torch.randn(2, sum(need), block, HKV, D, generator=g).to(torch.float8_e4m3fn)
        rows = codes.double() * torch.tensor([0.5, 2.0])[:, None, None, None, None]
        raw = codes.view(torch.uint8)
        for b, n in enumerate(lens):
            if n % block:
                raw[:, table[b, need[b] - 1], n % block:] = 0x7F   # NaN codes
        kw = dict(fp8_scales=(0.5, 2.0))
    dc = codes.to(dev)
    out = sb.ops.swa_decode_attention(q.to(dev), dc[0], dc[1], torch.tensor(lens, dtype=torch.int32, device=dev),
                                      block_table=table.to(dev), window_left=window, n_split=n_split, **kw)
    ref = []
    for b, n in enumerate(lens):
        k, v = rows[:, table[b, :need[b]].long()].flatten(1, 2)[:, max(0, n - 1 - window):n].repeat_interleave(HQ // HKV, 2)
        p = torch.softmax((q[b].double()[None] * k).sum(-1) * D ** -0.5, 0)
        ref.append((p[..., None] * v).sum(0))
    ref = torch.stack(ref)
    assert (out.cpu().double() - ref).abs().max() <= 2 ** -7 * ref.abs().max()
