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
    gate = torch.randn(64, 64, device=gpu)
    return lambda: plain.silu(gate, gate)


@pytest.mark.parametrize("op", ["decode", "prefill", "append", "silu"])
def test_other_threads_run_during_a_call(gpu, op):
    """The interpreter lock is free while a call allocates and launches. The
    switch interval is far above the test's length, so that another thread gets
    the lock only where this one gives it up. One call gives it up for a few
    microseconds, in which the waiting thread may or may not wake: 50000 calls at
    most are tried, until it has run. The outputs are kept meanwhile, since freeing a
    tensor may let go of the lock too."""
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
            outputs = [call() for _ in range(1000)]
            ran = count[0] != before
            del outputs
            if ran:
                break
    finally:
        stop.append(True)
        sys.setswitchinterval(interval)
        thread.join(5)
    assert ran


def tensors(op, gpu, dtype=torch.bfloat16):
    """Arguments of a plain call of the module's function."""
    if op == "decode":
        q, k, v, tables, lengths = random_paged([200, 64, 777], 8, 2, 64, dtype, gpu)
        return [q, k, v, tables, lengths, 0]
    if op == "prefill":
        return list(prefill_inputs([(500, 40), (77, 9), (30, 1)], 8, 2, 64, dtype, gpu))
    gen = torch.Generator().manual_seed(5)
    if op == "append":
        pools = [torch.randn(9, 16, 2, 64, generator=gen).to(dtype).to(gpu) for _ in range(2)]
        rows = [torch.randn(20, 2, 64, generator=gen).to(dtype).to(gpu) for _ in range(2)]
        at = torch.randperm(9 * 16, generator=gen)[:20].to(gpu)
        return pools + rows + [at // 16, at % 16]
    return [torch.randn(33, 71, generator=gen).to(dtype).to(gpu) for _ in range(2)]


def adapter(op):
    from vllm_rlt.kernels import activation, hip_attention

    return {"decode": hip_attention.paged_attention, "prefill": hip_attention.paged_prefill_attention,
            "append": hip_attention.kv_append, "silu": activation.silu_and_mul}[op]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("op", ["decode", "prefill", "append", "silu"])
def test_module_and_ctypes_paths_give_the_same_bits(gpu, op, dtype, monkeypatch):
    from vllm_rlt.kernels import activation, hip_attention
    from vllm_rlt.kernels._extension import plain_calls

    results = []
    for direct in (True, False):
        args = tensors(op, gpu, dtype)
        if direct:
            out = getattr(plain_calls(), op)(*args)
            assert out is not None  # the call is a plain one
            out = args[:2] if op == "append" else [out]
        else:
            for module in (hip_attention, activation):
                monkeypatch.setattr(module, "plain_calls", lambda: None)
            out = adapter(op)(*args)
            out = args[:2] if op == "append" else [out]
        results.append(out)
    assert all(torch.equal(a, b) for a, b in zip(*results))


class Subclass(torch.Tensor):
    pass


def replaced(args, index, value):
    return args[:index] + [value] + args[index + 1 :]


# Changes after which a call is not a plain one: (operations, change of the arguments).
DECLINED = {
    "subclass": ("decode prefill append silu", lambda a: replaced(a, 0, a[0].as_subclass(Subclass))),
    "cpu_tensor": ("decode prefill append silu", lambda a: replaced(a, 1, a[1].cpu())),
    "other_dtype": ("decode prefill append silu", lambda a: replaced(a, 1, a[1].double())),
    "not_a_tensor": ("decode prefill append silu", lambda a: replaced(a, 1, None)),
    "too_few": ("decode prefill append silu", lambda a: a[:-1]),
    "wider_tables": ("decode prefill", lambda a: replaced(a, 3, a[3].long())),
    "strided_lengths": ("decode prefill", lambda a: replaced(a, 4, a[4].repeat_interleave(2)[::2])),
    "long_lengths": ("decode prefill", lambda a: replaced(a, 4, a[4].long())),
    "heads_do_not_divide": ("decode prefill", lambda a: replaced(a, 0, a[0][:, :7])),
    "strided_head_dim": ("decode prefill", lambda a: replaced(a, 0, a[0].mT.contiguous().mT)),
    "no_rows": ("decode prefill", lambda a: replaced(a, 0, a[0][:0])),
    "rows_differ": ("decode", lambda a: replaced(a, 0, a[0][:2])),
    "bool_window": ("decode", lambda a: replaced(a, 5, True)),
    "negative_window": ("decode", lambda a: replaced(a, 5, -1)),
    "overlong_window": ("decode", lambda a: replaced(a, 5, 2**63)),
    "overlong_max_seqlen": ("prefill", lambda a: replaced(a, 6, 2**31)),
    "bounds_too_short": ("prefill", lambda a: replaced(a, 5, a[5][:-1])),
    "int_blocks": ("append", lambda a: replaced(a, 4, a[4].int())),
    "few_blocks": ("append", lambda a: replaced(a, 4, a[4][:-1])),
    "cache_layouts_differ": ("append", lambda a: replaced(
        a, 1, a[1].transpose(0, 1).contiguous().transpose(0, 1))),
    "transposed": ("silu", lambda a: [x.t() for x in a]),
    "gradient": ("silu", lambda a: replaced(a, 0, a[0].clone().requires_grad_())),
}


@pytest.mark.parametrize("op,change", [(op, name) for name, (ops, _) in DECLINED.items()
                                       for op in ops.split()])
def test_other_calls_are_left_to_the_adapter(gpu, op, change):
    from vllm_rlt.kernels._extension import plain_calls

    call = getattr(plain_calls(), op)
    args = tensors(op, gpu)
    pools = [x.clone() for x in args[:2]] if op == "append" else []
    assert call(*DECLINED[change][1](args)) is None
    assert all(torch.equal(a, b) for a, b in zip(args, pools))  # and wrote nothing


@pytest.mark.parametrize("op", ["decode", "prefill", "append", "silu"])
def test_calls_under_a_mode_are_left_to_the_adapter(gpu, op):
    from torch.overrides import TorchFunctionMode
    from torch.utils._python_dispatch import TorchDispatchMode

    from vllm_rlt.kernels._extension import plain_calls

    class Function(TorchFunctionMode):
        def __torch_function__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    class Dispatch(TorchDispatchMode):
        def __torch_dispatch__(self, func, types, args=(), kwargs=None):
            return func(*args, **(kwargs or {}))

    call = getattr(plain_calls(), op)
    args = tensors(op, gpu)
    for mode in (Function, Dispatch):
        with mode():
            assert call(*args) is None


@pytest.mark.parametrize("op,change,error", [
    ("decode", "negative_window", ValueError), ("decode", "bool_window", ValueError),
    ("decode", "wider_tables", ValueError), ("decode", "rows_differ", ValueError),
    ("prefill", "bounds_too_short", ValueError), ("append", "few_blocks", ValueError),
    ("silu", "cpu_tensor", ValueError)])
def test_what_the_adapter_refuses_stays_refused(gpu, op, change, error):
    with pytest.raises(error):
        adapter(op)(*DECLINED[change][1](tensors(op, gpu)))
