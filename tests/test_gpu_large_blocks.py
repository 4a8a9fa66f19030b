"""Paged caches with blocks of so many rows that the kernels' tile -> block multiplication exceeds the quotient: 46410 tiles
of 16 rows, where the last tile would be counted to the next block (and the block table read past its row). The same
memory seen as blocks of 16 rows gives the same bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
TILES, D = 46410, 128


@pytest.fixture(scope="module")
def cache(dev):
    """Codes and scales of one sequence, as one block."""
    g = torch.Generator(device=dev).manual_seed(0)
    rows = 16 * TILES
    codes = torch.randint(-127, 128, (2, 1, rows, 1, D), generator=g, device=dev, dtype=torch.int8)
    scales = torch.rand(2, 1, 1, rows, generator=g, device=dev) * 0.02 + 0.005
    return codes, scales


def _views(cache):
    codes, scales = cache
    dev = codes.device
    yield codes, scales, torch.zeros(1, 1, dtype=torch.int32, device=dev)
    yield codes.view(2, TILES, 16, 1, D), scales.view(2, TILES, 1, 16), torch.arange(TILES, dtype=torch.int32, device=dev)[None]


@pytest.mark.parametrize("hidden", [0, 16, 21])
def test_byte_code_decode(sb, dev, cache, hidden):
    q = torch.randn(1, 7, D, device=dev, generator=torch.Generator(device=dev).manual_seed(1)).bfloat16()
    lens = torch.tensor([16 * TILES - hidden], dtype=torch.int32, device=dev)
    one, many = (sb.ops.swa_decode_attention(q, c[0], c[1], lens, block_table=t, window_left=500, n_split=3, k_scale=s[0], v_scale=s[1])
                 for c, s, t in _views(cache))
    assert torch.equal(one, many)


def test_prompt_chunk(sb, dev, cache):
    q = torch.randn(40, 7, D, device=dev, generator=torch.Generator(device=dev).manual_seed(2)).bfloat16()
    one, many = (sb.ops.swa_prefill_attention(q, c[0], c[1], query_lens=[40], seq_lens_k=[16 * TILES], block_table=t, window_left=500,
                                              k_scale=s[0], v_scale=s[1]) for c, s, t in _views(cache))
    assert torch.equal(one, many)
