"""Small decode batches: split counts at the edges of the merge kernels' batches (4, 8 and, below 12, 16 partials per trip;
from 12 on 16, 32, 48 and 64 by four groups of threads), in fp32 against float64 attention (2e-6 of the largest value: 32-bit sums over at most 700 keys), and the bf16 stream kernel at
the split the library chooses against the same rows unsplit (both round fp32 results to bf16: one last place, 2^-7)."""
import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D, BS = 8, 2, 128, 16


def _problem(dev, dtype, lens, seed):
    g = torch.Generator().manual_seed(seed)
    need = [(n + BS - 1) // BS for n in lens]
    perm = torch.randperm(sum(need), generator=g).int()
    tables = torch.zeros(len(lens), max(need), dtype=torch.int32)
    at = 0
    for b, n in enumerate(need):
        tables[b, :n] = perm[at:at + n]
        at += n
    kv = torch.randn(2, sum(need), BS, HKV, D, generator=g).to(dtype)
    q = torch.randn(len(lens), HQ, D, generator=g).to(dtype)
    return q, kv, tables, torch.tensor(lens, dtype=torch.int32)


def _reference(q, kv, tables, lens, window):
    out = []
    for b, n in enumerate(lens):
        rows = kv[:, tables[b].long()].flatten(1, 2)[:, max(0, n - 1 - window):n].double()
        k, v = rows.repeat_interleave(HQ // HKV, dim=2).unbind(0)
        p = torch.softmax(torch.einsum("hd,khd->hk", q[b].double(), k) * D ** -0.5, -1)
        out.append(torch.einsum("hk,khd->hd", p, v))
    return torch.stack(out)


@pytest.mark.parametrize("n_split", [2, 4, 5, 8, 9, 11, 12, 13, 15, 16, 17, 31, 32, 33, 47, 48, 49, 63, 64, 65, 130])
def test_merge_of_many_partials(sb, dev, n_split):
    lens = [700, 33, 1, 512, 97]          # rows with fewer chunks than splits leave empty partials
    q, kv, tables, sl = _problem(dev, torch.float32, lens, n_split)
    kvd = kv.to(dev)
    out, lse = sb.ops.swa_decode_attention(q.to(dev), kvd[0], kvd[1], sl.to(dev), block_table=tables.to(dev), window_left=650,
                                           n_split=n_split, balanced=False, return_lse=True)
    ref = _reference(q, kv, tables, lens, 650)
    assert (out.cpu().double() - ref).abs().max() <= 2e-6 * ref.abs().max() and torch.isfinite(lse).all()


@pytest.mark.parametrize("rows", [1, 3, 17])
@pytest.mark.parametrize("length", [350, 353, 600, 1000, 2048])
def test_chosen_split_matches_unsplit_rows(sb, dev, rows, length):
    lens = [max(1, length - 37 * i) for i in range(rows)]
    q, kv, tables, sl = _problem(dev, torch.bfloat16, lens, length)
    q, kv, tables, sl = q.to(dev), kv.to(dev), tables.to(dev), sl.to(dev)
    assert sb._native.lib().sb_swa_decode_auto_split(rows, HKV, tables.shape[1] * BS, 1024) > 1
    one, auto = (sb.ops.swa_decode_attention(q, kv[0], kv[1], sl, block_table=tables, window_left=1024, n_split=n, balanced=False)
                 for n in (1, 0))
    assert ((auto.float() - one.float()).abs() <= 2 ** -7 * one.float().abs() + 2 ** -9 * one.float().abs().max()).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("how", [dict(n_split=n, balanced=False) for n in (2, 3, 5, 9, 10, 13)] + [
    dict(n_split=3, merge_in_kernel=True, balanced=False), dict(n_split=3, balanced=True), dict(n_split=3, balanced=True, per_segment=True)])
def test_infinite_value_in_the_last_partial(sb, dev, dtype, how):
    """A visible key whose value is infinite makes the output infinite however the row is cut: the merges fill the
    rest of a trip to memory with the last partial again, which must not count (infinity times 0 is a NaN)."""
    if dtype == torch.float32 and (how["balanced"] or "merge_in_kernel" in how):
        pytest.skip("matrix-core kernels only")
    lens = [320, 320]
    q, kv, tables, sl = _problem(dev, dtype, lens, 4)
    kv[1, tables[0, 19], 15, :, 5] = float("inf")     # the newest key of row 0
    kvd = kv.to(dev)
    run = lambda **kw: sb.ops.swa_decode_attention(q.to(dev), kvd[0], kvd[1], sl.to(dev), block_table=tables.to(dev),
                                                   window_left=1024, **kw).float().cpu()
    whole, cut = run(n_split=1, balanced=False), run(**how)
    assert torch.isposinf(whole[0, :, 5]).all() and torch.isposinf(cut[0, :, 5]).all()
    assert torch.equal(torch.isfinite(whole), torch.isfinite(cut))
