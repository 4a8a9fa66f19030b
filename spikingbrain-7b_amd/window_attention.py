"""Cache + attention slice of the HuggingFace-side sliding-window layer.

Mirrors the part of `FlashAttention.forward` between RoPE and `o_proj`:
  hf_7B_model/window_attention.py:164-217      (flash flavour: window_size=(W, 0), i.e. the query
                                                sees itself and W keys to its left)
  hf_7B_model/window_attention_sdpa.py:174-214 (SDPA flavour: W keys including itself, and no
                                                window_size handed to the cache, :176)
Projections, RoPE and o_proj stay with the caller; inputs are the post-RoPE q/k/v.
"""
from __future__ import annotations

from typing import Optional

import torch

from . import ops
from .hf_cache import Cache


# query runs at least this long use the many-query kernel; shorter ones (speculative / multi-token
# decode) run as rows of the single-query kernel, which wastes no tile rows on them
PREFILL_MIN_QUERIES = 16

_plans: dict = {}


def _uniform_plan(B: int, Q: int, K: int, dev: torch.device):
    """Tile plan for B sequences of Q queries over K keys each (every layer of a forward pass asks
    for the same one)."""
    key = (B, Q, K, dev)
    plan = _plans.get(key)
    if plan is None:
        if len(_plans) >= 64:
            _plans.clear()
        plan = _plans[key] = ops.PrefillPlan([Q] * B, [K] * B, dev)
    return plan


def _kv_step_rows(k: torch.Tensor) -> Optional[int]:
    """Distance of two batch entries in units of k.stride(2); None if it is not a whole number."""
    if k.shape[0] == 1:
        return 0
    if k.stride(2) == 0 or k.stride(0) % k.stride(2) != 0:
        return None
    return k.stride(0) // k.stride(2)


def sliding_window_attention(
    query_states: torch.Tensor,
    key_states: torch.Tensor,
    value_states: torch.Tensor,
    sliding_window: int,
    past_key_values: Optional[Cache] = None,
    layer_idx: int = 0,
    attention_mask: Optional[torch.Tensor] = None,
    flavour: str = "flash",
    cache_window_size: Optional[int] = -1,
    window_left: Optional[int] = None,
) -> torch.Tensor:
    """query_states [B, Hq, Q, D]; key_states/value_states [B, Hkv, Q, D] (new tokens only).
    Appends the new K/V to `past_key_values` exactly as the reference layer does, then attends
    causally inside the sliding window over the cached (or, on the first call, the in-flight)
    keys. `attention_mask` [B, >=K] marks left padding with 0. Returns [B, Q, Hq, D].
    `flavour` picks the two conventions the reference files use (flash: cache bounded at W rows,
    W keys left of the query visible; sdpa: cache unbounded, W keys including the query);
    `cache_window_size` (None = unbounded) and `window_left` override them one by one, e.g. a
    bounded cache with the SDPA mask.
    A fully masked query row (a pad position) comes out as zeros."""
    if flavour not in ("flash", "sdpa"):
        raise ValueError("flavour must be 'flash' or 'sdpa'")
    B, Hq, Q, D = query_states.shape
    if window_left is None:
        window_left = sliding_window if flavour == "flash" else sliding_window - 1
    # one new token of a few sequences, in a form that the native step has (ops.dense_decode, which would turn the others down at
    # 2 us a call)
    one_step = Q == 1 and D == 128 and B <= 64 and query_states.is_cuda and Hq <= 16 * key_states.shape[1] and \
        (attention_mask is None or not attention_mask.dtype.is_floating_point)
    if past_key_values is not None:
        cache_has_content = past_key_values.get_seq_length(layer_idx) > 0
        if cache_window_size == -1:
            cache_kwargs = {"window_size": sliding_window} if flavour == "flash" else {}
        else:
            cache_kwargs = {"window_size": cache_window_size}
        if one_step and cache_has_content and type(past_key_values) is Cache and \
                getattr(past_key_values.update, "__func__", None) is _UPDATE:
            return _decode_step(past_key_values, layer_idx, query_states, key_states, value_states, attention_mask, window_left, cache_kwargs)
        key_cached, value_cached = past_key_values.update(
            attn_state=(key_states, value_states), layer_idx=layer_idx, offset=Q,
            cache_kwargs=cache_kwargs)["attn_state"]
        if cache_has_content:
            key_states, value_states = key_cached, value_cached

    if one_step:
        out = ops.dense_decode(query_states, key_states, value_states, attention_mask, window_left, D ** -0.5)
        if out is not None:
            return out
    return _attend(query_states, key_states, value_states, attention_mask, window_left)


_UPDATE = Cache.update   # (a cache with another one is updated through that)


def _decode_step(cache: Cache, layer_idx: int, q, key, value, mask, window_left: int, cache_kwargs) -> torch.Tensor:
    """One new token against a cache that has rows: their copy into the window goes with the attention's first launch. Refused rows leave
    the cache as it was; where the rows are fine and the attention fails, they are in the cache, as after an `update` by itself."""
    out = failure = None

    def push(k_copy, v_copy, rows):
        nonlocal out, failure
        try:
            out = ops.dense_decode(q, *rows, mask, window_left, q.shape[3] ** -0.5, (k_copy, v_copy))
        except Exception as e:
            failure = e
        if out is None:
            ops.window_shift_pair(k_copy, v_copy)

    rows = cache._update(push, None, (key, value), None, layer_idx, 1, cache_kwargs)["attn_state"]
    if failure is not None:
        raise failure
    return out if out is not None else _attend(q, *rows, mask, window_left)


def _attend(query_states, key_states, value_states, attention_mask, window_left: int) -> torch.Tensor:
    """The queries [B, Hq, Q, D] are the last Q of the keys' [B, Hkv, K, D] positions; returns [B, Q, Hq, D]."""
    B, Hq, Q, D = query_states.shape
    Hkv, K = key_states.shape[1], key_states.shape[2]
    k, v = key_states, value_states
    if k.stride(3) != 1 or v.stride() != k.stride() or _kv_step_rows(k) is None:
        k, v = k.contiguous(), v.contiguous()

    q_rows = query_states.transpose(1, 2).reshape(B * Q, Hq, D)
    dev = q_rows.device
    # left padding: zeros form a prefix of a sequence's mask
    keep = None if attention_mask is None else attention_mask[:, -K:]
    pad = None
    if keep is not None and keep.dim() != 2:
        pad, keep = (K - (keep != 0).sum(dim=1)).to(torch.int32).contiguous(), None
    if Q >= PREFILL_MIN_QUERIES and q_rows.dtype in (torch.bfloat16, torch.float16) and D == 128:
        # prompt-sized query runs go to the matrix-core kernel (64-token tiles): one bound per sequence
        _, _, key_lo, kv_start = ops.dense_rows(B, 1, K, _kv_step_rows(k), dev, keep)
        out = ops.swa_prefill_attention(
            q_rows, k, v, plan=_uniform_plan(B, Q, K, dev), kv_start=kv_start, key_lo=key_lo if pad is None else pad,
            kv_strides=(k.stride(2), k.stride(1)), num_kv_heads=Hkv, window_left=window_left, scale=D ** -0.5)
        return out.view(B, Q, Hq, D)
    seq_lens_row, row_seq, key_lo, kv_start = ops.dense_rows(B, Q, K, _kv_step_rows(k), dev, keep)
    if pad is not None:
        key_lo = pad.repeat_interleave(Q)
    out = ops.swa_decode_attention(
        q_rows, k, v, seq_lens_row, kv_start=kv_start, row_seq=row_seq, key_lo=key_lo,
        kv_strides=(0, k.stride(2), k.stride(1)), num_kv_heads=Hkv, window_left=window_left,
        scale=D ** -0.5, max_seq_len=K)
    return out.view(B, Q, Hq, D)
