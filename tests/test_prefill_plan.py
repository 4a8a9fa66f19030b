"""Tile plans of the prompt kernel (host only)."""
import ctypes
import random

import pytest


@pytest.mark.parametrize("lens_q,lens_k", [([64], [2**32 + 64]), ([1], [2**31]), ([5, 64], [5, 2**31 + 7]), ([2**30, 2**30], None)])
def test_lengths_beyond_32_bits_are_refused(sb, lens_q, lens_k):
    """The kernel reads 32-bit lengths; a wrapped one would be another length (or a negative one)."""
    with pytest.raises(RuntimeError, match="without overflow"):
        sb.ops.PrefillPlan(lens_q, lens_k, "cpu")


def test_longest_length_that_fits(sb):
    plan = sb.ops.PrefillPlan([1], [2**31 - 1], "cpu")
    assert plan.seq_lens_k.tolist() == [2**31 - 1] and plan.max_k == 2**31 - 1


def _lists(lens, keys):
    """The tiles of a list of less than 1024: latest in the keys first, dealt to the eighths of the list in turn."""
    tiles = [(s, at) for s, n in enumerate(lens) for at in range(0, n, 64)]
    tiles.sort(key=lambda t: -(t[1] + keys[t[0]] - lens[t[0]]))
    per = -(-len(tiles) // 8)
    slots = [k % 8 * per + k // 8 for k in range(8 * per)]
    return [t for _, t in sorted(zip([x for x in slots if x < len(tiles)], tiles))]


def test_dealt_lists(sb):
    rng = random.Random(0)
    cases = [[64 * t - rng.randint(0, 63)] for t in list(range(1, 70)) + [127, 128, 129, 1023]] + [[], [0], [0, 5, 0]]
    cases += [[rng.choice([0, 1, rng.randint(1, 700)]) for _ in range(rng.randint(1, 12))] for _ in range(200)]
    for lens in cases:
        keys = [n + rng.choice([0, 0, rng.randint(0, 6000)]) for n in lens]
        plan = sb.ops.PrefillPlan(lens, keys, "cpu")
        assert list(zip(plan.tile_seq.tolist(), plan.tile_q0.tolist())) == _lists(lens, keys), (lens, keys)


def test_long_lists_keep_sequence_order(sb):
    lens = [64 * 700, 1, 64 * 323]
    plan = sb.ops.PrefillPlan(lens, None, "cpu")
    assert plan.num_tiles == 1024
    assert list(zip(plan.tile_seq.tolist(), plan.tile_q0.tolist())) == [(s, at) for s, n in enumerate(lens) for at in range(0, n, 64)]


def test_native_plan_refuses_what_does_not_fit(sb):
    L, ints = sb._native.lib(), ctypes.c_int32 * 2
    plan = (ctypes.c_int32 * 64)()
    run = lambda q, k, tiles: L.sb_swa_prefill_plan(ints(*q), ints(*k), 2, tiles, ctypes.addressof(plan))
    assert run((64, 65), (64, 65), 3) == 0 and list(plan[:5]) == [0, 64, 129, 64, 65]
    for q, k, tiles in (((64, 65), (64, 65), 2), ((64, 65), (64, 65), 4), ((64, 65), (64, 64), 3), ((-1, 65), (64, 65), 2)):
        assert run(q, k, tiles) == sb._native.SB_ERR_INVALID
    assert L.sb_swa_prefill_plan(None, None, 1, 1, ctypes.addressof(plan)) == sb._native.SB_ERR_INVALID


@pytest.mark.parametrize("lens", [[64], [1517, 3, 900], [100] * 128, [100] * 129, [8192] * 2, [8192] * 16])
def test_plan_covers_every_tile_once(sb, lens):
    plan = sb.ops.PrefillPlan(lens, [n + 7 for n in lens], "cpu")
    want = [(s, at) for s, n in enumerate(lens) for at in range(0, n, 64)]
    assert sorted(zip(plan.tile_seq.tolist(), plan.tile_q0.tolist())) == want and plan.num_tiles == len(want)
    assert plan.cu_seqlens_q.tolist() == [sum(lens[:i]) for i in range(len(lens) + 1)]
    assert plan.seq_lens_k.tolist() == [n + 7 for n in lens] and plan.total_k == sum(lens) + 7 * len(lens)
    assert all(t.dtype == plan.cu_seqlens_q.dtype for t in (plan.seq_lens_k, plan.tile_seq, plan.tile_q0))
