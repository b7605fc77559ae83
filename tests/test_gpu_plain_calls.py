"""The extension module's one-step functions (decode, prefill, append, SiLU-and-Mul)
that the adapter tries first: what they may hold up while they run."""

import sys
import threading
import time

import pytest
import torch

from test_gpu_attention import prefill_inputs, random_paged

pytestmark = pytest.mark.gpu


def plain_call(op, gpu):
    """A call of the module itself."""
    from vllm_rlt.kernels._extension import plain_calls

    plain = plain_calls()
    if op == "decode":
        q, k, v, tables, lengths = random_paged([200] * 64, 16, 16, 128, torch.bfloat16, gpu)
        return lambda: plain.decode(q, k, v, tables, lengths, 0)
    if op == "prefill":
        inputs = prefill_inputs([(1500, 300)], 16, 16, 128, torch.bfloat16, gpu)
        return lambda: plain.prefill(*inputs)
    if op == "append":
        pool = torch.zeros(64, 16, 16, 128, dtype=torch.bfloat16, device=gpu)
        rows = torch.randn(1024, 16, 128, device=gpu).to(torch.bfloat16)
        at = torch.arange(1024, device=gpu)
        args = (pool, pool.clone(), rows, rows, at // 16, at % 16)
        return lambda: plain.append(*args)
    gate = torch.randn(4096, 4096, device=gpu)
    return lambda: plain.silu(gate, gate)


@pytest.mark.parametrize("op", ["decode", "prefill", "append", "silu"])
def test_other_threads_run_during_a_call(gpu, op):
    """The interpreter lock is free while a call allocates and launches. The
    switch interval is far above the test's length, so that another thread gets
    the lock only where this one gives it up. One call gives it up for a few
    microseconds, in which the waiting thread may or may not wake: 50000 calls at
    most are tried, until it has run."""
    call = plain_call(op, gpu)
    assert call() is not None
    count, stop = [0], []

    def other():
        while not stop:
            count[0] += 1
            time.sleep(0)

    thread = threading.Thread(target=other, daemon=True)
    interval = sys.getswitchinterval()
    sys.setswitchinterval(1000)
    ran = False
    try:
        thread.start()
        for _ in range(50):
            torch.cuda.synchronize()
            before = count[0]
            for _ in range(1000):
                call()
            # Nothing between these two lines but the calls lets go of the lock.
            ran = count[0] != before
            if ran:
                break
    finally:
        stop.append(True)
        sys.setswitchinterval(interval)
        thread.join(5)
    assert ran
