"""How a prompt call is spread over the GPU (256 CUs where the device cannot be asked): parts of the walks side by side, halves of them in
one workgroup, or neither, for calls whose times lie 5 % or more apart. us as measured: in parts, in halves, in groups of three or four heads."""
import ctypes

import pytest


@pytest.mark.parametrize("hq,hkv,lens,context,window,parts,halves", [
    (8, 4, [2048], 2000, 4096, True, True),         # 59.8, 69.4
    (8, 4, [700], 2000, 1024, True, True),          # 20.5, 26.4
    (16, 8, [400], 800, 4096, True, True),          # 21.1, 27.5
    (4, 2, [3000], 800, 4096, True, True),          # 55.0, 64.7
    (12, 4, [2048], 2000, 4096, True, True),        # 66, 71.5
    (6, 2, [4096], 0, 4096, True, True),            # 65.5, 70.7
    (28, 4, [1024], 10000, 4096, False, True),      # 79.7, 74.1
    (28, 4, [512], 10000, 4096, True, True),        # 52, 72.6
    (28, 4, [64], 10000, 4096, True, True),         # 26, 69
    (12, 4, [1088], 2000, 4096, True, True),        # 44.1, 55.6
    (16, 4, [1517], 0, 4096, False, True),          # 33.8, 30.7
    (28, 4, [1517], 0, 4096, False, True),          # 44.6, 34.3
    (12, 4, [3000], 2000, 4096, False, False),      # halves 111.6, groups of three 105
    (24, 8, [1517], 2000, 4096, False, False),      # halves 95.9, groups of three 88.2
    (18, 6, [1517], 2000, 4096, False, True),       # halves 75.6, groups of three 90.3
    (28, 4, [2048], 10000, 4096, False, False),     # halves 149, groups of four 132
])
def test_parts_or_halves(sb, hq, hkv, lens, context, window, parts, halves):
    """`parts`: the call is cut into several; `halves`: what a call that is not cut does."""
    plan = sb.ops.PrefillPlan(lens, [n + context for n in lens], "cpu")
    a = sb._native.SwaPrefillArgs(num_tiles=plan.num_tiles, num_q_heads=hq, num_kv_heads=hkv, window_left=window, tile_keys=plan.tile_keys_ptr)
    L = sb._native.lib()
    assert (L.sb_swa_prefill_parts(ctypes.byref(a), plan.max_k) > 1) == parts
    assert L.sb_swa_prefill_halves(ctypes.byref(a), plan.max_k, 1) == halves
    assert L.sb_swa_prefill_halves(ctypes.byref(a), plan.max_k, 2) == 0
    if halves:
        assert L.sb_swa_prefill_group_heads(ctypes.byref(a), plan.max_k, 1) == 2


def test_no_halves_without_tiles_or_beside_meta_rows(sb):
    L, args = sb._native.lib(), sb._native.SwaPrefillArgs
    assert L.sb_swa_prefill_halves(None, 100, 1) == 0 and L.sb_swa_prefill_halves(ctypes.byref(args()), 100, 1) == 0
    a = args(num_tiles=8, num_q_heads=28, num_kv_heads=4, window_left=4096, meta_len=16)
    assert L.sb_swa_prefill_halves(ctypes.byref(a), 512, 1) == 0
    a.meta_len = 0
    assert L.sb_swa_prefill_halves(ctypes.byref(a), 512, 1) == 1
