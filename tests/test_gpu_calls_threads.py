"""The native layer calls let go of the interpreter lock while they allocate and launch."""
import sys
import threading
import time

import pytest
import torch

pytestmark = pytest.mark.gpu
HQ, HKV, D = 4, 2, 128


def _recorded(sb, monkeypatch, run):
    """The native calls that run() makes, as (name, function, arguments)."""
    real, seen = sb._native.calls(), []

    class Record:
        def __getattr__(self, name):
            return lambda *a: seen.append((name, getattr(real, name), a)) or getattr(real, name)(*a)

    with monkeypatch.context() as m:
        m.setattr(sb._native, "calls", lambda: Record())
        run()
    return seen


def _layer_calls(sb, dev):
    rand = lambda *s: torch.randn(*s, device=dev).bfloat16()
    cache, table = rand(2, 8, 16, HKV, D), torch.arange(8, dtype=torch.int32, device=dev).view(2, 4)
    lens, slots = torch.tensor([50, 20], dtype=torch.int32, device=dev), torch.tensor([49, 83], device=dev)
    q, k, v = rand(2, HQ, D), rand(2, HKV, D), rand(2, HKV, D)
    sb.ops.kv_append(k, v, cache[0], cache[1], slots)
    sb.ops.swa_decode_attention(q, cache[0], cache[1], lens, block_table=table, window_left=63, out=torch.empty_like(q), balanced=False)
    sb.ops.fp8_step(None, [(q, 1.0)])
    plan = sb.ops.PrefillPlan([2], [2], dev)
    sb.ops.swa_prefill_attention(q, k, v, plan=plan, out=torch.empty_like(q), kv_start32=torch.zeros(1, dtype=torch.int32, device=dev))
    sb.my_fused_recurrent_gla(q[:, :, None], *(rand(2, HQ, 1, D) for _ in range(2)), -torch.rand(2, HQ, 1, D, device=dev), torch.zeros(2, HQ, D, D, device=dev), None)
    hf = sb.Cache()
    hf.update(attn_state=(rand(2, HKV, 8, D), rand(2, HKV, 8, D)), layer_idx=0, offset=8, cache_kwargs={"window_size": 8})
    hf.update(attn_state=(rand(2, HKV, 1, D), rand(2, HKV, 1, D)), layer_idx=0, offset=1, cache_kwargs={"window_size": 8})
    sb.sliding_window_attention(q[:, :, None], k[:, :, None], v[:, :, None], 8, hf, 0)
    return plan


def test_other_threads_run_during_a_call(sb, dev, monkeypatch):
    """With a switch interval that never comes, a second thread gets the interpreter only where the first one lets go of it."""
    kept = []
    _layer_calls(sb, dev)                                                  # (scratch memory, lazy imports)
    calls = _recorded(sb, monkeypatch, lambda: kept.append(_layer_calls(sb, dev)))
    calls = [c for c in calls if c[0] != "decodes"]                         # (asks about tensors, launches nothing)
    assert {n for n, _, _ in calls} == {"append", "decode", "append_fp8", "prefill", "gla_step", "push", "dense_decode"}
    count, stop, started = [0], [], threading.Event()

    def other():
        started.set()
        while not stop:
            count[0] += 1
            time.sleep(0)

    interval = sys.getswitchinterval()
    thread = threading.Thread(target=other)
    try:
        sys.setswitchinterval(1000)
        thread.start()
        started.wait()
        stuck = []
        for name, function, args in calls:
            before = count[0]
            for _ in range(10000):
                function(*args)
                if count[0] != before:
                    break
            else:
                stuck.append(name)
    finally:
        stop.append(1)
        sys.setswitchinterval(interval)
        thread.join()
        torch.cuda.synchronize()
    assert not stuck
