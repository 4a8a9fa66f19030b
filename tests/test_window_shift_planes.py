"""Where window_shift finds the new rows of a cache layer, [B, H, n, D] as a projection leaves them ([B, n, H, D] transposed, among them one
kv head, whose rows count as contiguous with any stride between heads), sliced or contiguous."""
import pytest
import torch

FORMS = {
    "transposed": lambda B, H, n, D, new: new(B, n, H, D).transpose(1, 2),
    "fused": lambda B, H, n, D, new: new(B, n, 3 * H, D)[:, :, H:2 * H].transpose(1, 2),
    "contiguous": lambda B, H, n, D, new: new(B, H, n, D),
    "sliced": lambda B, H, n, D, new: new(B, H, n + 3, D)[:, :, 2:2 + n],
}
SIZES = [(1, 1, 1), (1, 1, 5), (1, 3, 5), (2, 1, 5), (3, 1, 1), (3, 1, 2), (3, 2, 1), (2, 4, 7)]


@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("B,H,n", SIZES)
def test_addresses(sb, monkeypatch, form, B, H, n):
    monkeypatch.setattr(sb.ops.N, "require_gpu", lambda *a: torch.device("cpu"))
    monkeypatch.setattr(sb.ops.N, "stream_ptr", lambda dev: 0)
    rows = FORMS[form](B, H, n, 16, lambda *shape: torch.randn(shape, generator=torch.Generator().manual_seed(n)))
    src, dst = (torch.zeros(B, m, H, 16).transpose(1, 2) if H == 1 else torch.zeros(B, H, m, 16) for m in (4, n + 2))   # (contiguous both ways)
    a, held = sb.ops._window_shift_args(src, dst, rows, 1, 0, 1)
    assert a.fresh == held.data_ptr() and a.planes == B * H and a.n_new == n
    assert (a.src_stride_plane_bytes, a.dst_stride_plane_bytes) == (4 * 16 * 4, (n + 2) * 16 * 4)
    got = torch.as_strided(held, (B * H, n, 16), (a.fresh_stride_plane_bytes // 4, a.fresh_stride_row_bytes // 4, 1), held.storage_offset())
    assert torch.equal(got, rows.reshape(B * H, n, 16))


@pytest.mark.gpu
@pytest.mark.parametrize("form", FORMS)
@pytest.mark.parametrize("B,H,n", SIZES)
def test_cache_rows(sb, dev, form, B, H, n):
    new = lambda seed: FORMS[form](B, H, n, 128, lambda *shape: torch.randn(shape, generator=torch.Generator().manual_seed(seed)).bfloat16().to(dev))
    cache, seen = sb.Cache(), []
    for step in range(3):
        k, v = new(2 * step), new(2 * step + 1)
        seen.append((k, v))
        rows = cache.update(attn_state=(k, v), layer_idx=0, offset=n, cache_kwargs={})["attn_state"]
        assert all(torch.equal(rows[i], torch.cat([x[i] for x in seen], 2)) for i in range(2))
