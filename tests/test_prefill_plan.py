"""Tile plans of the prompt kernel (host only)."""
import copy
import ctypes
import pickle
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
        T, at = plan.num_tiles, 2 * len(lens) + 1
        ordered = plan._host[at + 2 * T:at + 4 * T].tolist()
        assert list(zip(ordered[:T], ordered[T:])) == [(s, q0) for s, n in enumerate(lens) for q0 in range(0, n, 64)]
        first = plan._host.data_ptr() + 4 * at
        assert plan.list_ptrs() == ((first + 16 * T, first + 8 * T, first + 12 * T) if T > 1 else (None, None, None))


def test_long_lists_keep_sequence_order(sb):
    lens = [64 * 700, 1, 64 * 323]
    plan = sb.ops.PrefillPlan(lens, None, "cpu")
    assert plan.num_tiles == 1024 and plan.list_ptrs() == (None, None, None)
    assert list(zip(plan.tile_seq.tolist(), plan.tile_q0.tolist())) == [(s, at) for s, n in enumerate(lens) for at in range(0, n, 64)]


def test_native_plan_refuses_what_does_not_fit(sb):
    L, ints = sb._native.lib(), ctypes.c_int32 * 2
    plan = (ctypes.c_int32 * 64)()
    run = lambda q, k, tiles: L.sb_swa_prefill_plan(ints(*q), ints(*k), 2, tiles, ctypes.addressof(plan), None)
    assert run((64, 65), (64, 65), 3) == 0 and list(plan[:5]) == [0, 64, 129, 64, 65]
    for q, k, tiles in (((64, 65), (64, 65), 2), ((64, 65), (64, 65), 4), ((64, 65), (64, 64), 3), ((-1, 65), (64, 65), 2)):
        assert run(q, k, tiles) == sb._native.SB_ERR_INVALID
    assert L.sb_swa_prefill_plan(None, None, 1, 1, ctypes.addressof(plan), None) == sb._native.SB_ERR_INVALID


@pytest.mark.parametrize("lens", [[64], [1517, 3, 900], [100] * 128, [100] * 129, [8192] * 2, [8192] * 16])
def test_plan_covers_every_tile_once(sb, lens):
    plan = sb.ops.PrefillPlan(lens, [n + 7 for n in lens], "cpu")
    want = [(s, at) for s, n in enumerate(lens) for at in range(0, n, 64)]
    assert sorted(zip(plan.tile_seq.tolist(), plan.tile_q0.tolist())) == want and plan.num_tiles == len(want)
    assert plan.cu_seqlens_q.tolist() == [sum(lens[:i]) for i in range(len(lens) + 1)]
    assert plan.seq_lens_k.tolist() == [n + 7 for n in lens] and plan.total_k == sum(lens) + 7 * len(lens)
    assert all(t.dtype == plan.cu_seqlens_q.dtype for t in (plan.seq_lens_k, plan.tile_seq, plan.tile_q0))


def _heads(sb, lens, context, window, known=True):
    """Query heads per workgroup of an uncut call of 28 : 4 heads (256 CUs where the device cannot be asked)."""
    keys = [n + context for n in lens]
    plan = sb.ops.PrefillPlan(lens, keys, "cpu")
    a = sb._native.SwaPrefillArgs(num_tiles=plan.num_tiles, num_q_heads=28, num_kv_heads=4, window_left=window,
                                  tile_keys=plan.tile_keys_ptr if known else None)
    return sb._native.lib().sb_swa_prefill_group_heads(ctypes.byref(a), plan.max_k, 1)


@pytest.mark.parametrize("lens,context,window,heads", [
    ([563], 4200, 4096, 2), ([1024], 4200, 4096, 2),                            # a workgroup of two heads for every CU
    ([1075], 4200, 512, 4), ([1523], 4200, 1024, 4), ([2035], 4200, 1024, 4), ([2035], 4200, 4096, 4), ([1000, 300, 600], 4200, 2048, 4),
    ([1075], 0, 512, 2), ([1523], 0, 512, 2), ([2035], 0, 512, 4),              # whole prompts, more and more walks of a full window
    ([1523], 0, 1024, 2), ([2035], 0, 4096, 2), ([1200], 300, 4096, 2), ([2000], 800, 4096, 2),
    ([3059], 4200, 1024, 2), ([3059], 4200, 4096, 4), ([3059], 0, 4096, 2), ([700] * 3, 0, 512, 2), ([6000], 0, 4096, 4)])
def test_heads_per_workgroup(sb, lens, context, window, heads):
    """Prompt chunks behind a context walk equally many keys per tile, whatever the window: above one workgroup of two heads
    per CU they take groups of four."""
    assert _heads(sb, lens, context, window) == heads
    tiles = sum(-(-n // 64) for n in lens)
    if 16 < tiles <= 32:
        assert _heads(sb, lens, context, window, known=False) == 4


def test_keys_of_the_tiles(sb):
    lens, keys = [100, 0, 64, 200], [100, 7, 3064, 250]
    plan = sb.ops.PrefillPlan(lens, keys, "cpu")
    got = plan._host[-plan.num_tiles:].tolist()
    assert got == sorted((64 + at + k - n for n, k in zip(lens, keys) for at in range(0, n, 64)), reverse=True)
    assert sb.ops.PrefillPlan([64 * 1024], None, "cpu").tile_keys_ptr is None


@pytest.mark.parametrize("again", [copy.copy, copy.deepcopy, lambda plan: pickle.loads(pickle.dumps(plan))])
def test_copies_do_not_read_the_original(sb, again):
    """A copied or saved plan outlives the one it was made of, and the call reads the tiles' keys on the host: from the
    copy's own memory, or not at all."""
    plan = sb.ops.PrefillPlan([100, 7, 640], [300, 7, 641], "cpu")
    host, keys = plan._host.data_ptr(), plan._host[-plan.num_tiles:].tolist()
    kept = again(plan)
    at = kept.tile_keys_ptr
    assert at is None or list((ctypes.c_int32 * kept.num_tiles).from_address(at)) == keys
    assert at is None or at == kept._host.data_ptr() + 4 * (kept._host.numel() - kept.num_tiles)
    if again is not copy.copy:
        assert kept._host.data_ptr() != host
    assert kept.tile_seq.tolist() == plan.tile_seq.tolist() and kept.tile_q0.tolist() == plan.tile_q0.tolist()


def test_lists_of_the_callers_own_have_no_known_keys(sb):
    plan = sb.ops.PrefillPlan([100, 7, 640], None, "cpu")
    assert plan.tile_keys_ptr is not None
    plan.num_tiles += 1
    assert plan.tile_keys_ptr is None
    plan.num_tiles -= 1
    plan.tile_q0 = plan.tile_q0.clone()
    assert plan.tile_keys_ptr is None
