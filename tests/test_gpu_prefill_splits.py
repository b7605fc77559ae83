"""Packed prefill with key splits: calls whose query tiles leave the GPU partly
idle cut each tile's keys into runs and merge the runs' fp32 partials. Checked
against the per-query oracle (tolerances of test_gpu_attention) where splitting
can go wrong: tile and run remainders, tiles shared by a group of q heads that
does not divide 128, sequences with fewer runs than the longest one, tiles that
see no key, both grid orders (kv heads a multiple of 8, and not), and partials
that nothing has initialised.
"""

import pytest
import torch

from test_gpu_attention import assert_close, oracle_prefill, prefill_inputs

pytestmark = pytest.mark.gpu

# (context, queries) per sequence; every batch has over 8 queries somewhere, so
# that it runs on the MFMA tiles, and few enough tiles to be split.
BATCHES = {
    "lone_chunk": [(1500, 129)],
    "lone_short": [(1411, 9)],
    "one_query_over": [(700, 33), (641, 32)],
    "ragged": [(1000, 64), (40, 40), (130, 17), (5, 5), (300, 1)],
    "no_visible_key": [(3, 20), (900, 10)],
}


def call(lib, inputs, nbytes, fill=0xFF):
    from vllm_rlt.kernels.hip_attention import dtype_code

    q, k, v, tables, lengths, cu, max_q = inputs
    out = torch.empty_like(q)
    workspace = torch.full((nbytes,), fill, dtype=torch.uint8, device=q.device)
    lib.check(lib.vrh_paged_prefill(
        dtype_code(q.dtype), out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        tables.data_ptr(), lengths.data_ptr(), cu.data_ptr(), len(lengths), q.shape[0], max_q,
        q.shape[1], k.shape[2], q.shape[2], k.shape[1], tables.shape[1], tables.stride(0),
        q.stride(0), q.stride(1), out.stride(0), out.stride(1), *k.stride()[:3], *v.stride()[:3],
        workspace.data_ptr(), nbytes, torch.cuda.current_stream().cuda_stream), "vrh_paged_prefill")
    return out


def sizes(lib, inputs):
    q, k, _, tables, lengths, _, max_q = inputs
    base = lib.vrh_paged_prefill_workspace_bytes(len(lengths), max_q, q.shape[1], q.shape[2])
    full = lib.vrh_paged_prefill_split_workspace_bytes(
        len(lengths), q.shape[0], max_q, q.shape[1], k.shape[2], q.shape[2], k.shape[1],
        tables.shape[1])
    return base, full


@pytest.mark.parametrize("batch", BATCHES)
@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim", [
    (torch.bfloat16, 8, 8, 128), (torch.bfloat16, 12, 4, 128), (torch.float16, 32, 8, 64),
    (torch.bfloat16, 5, 1, 96), (torch.float16, 2, 2, 32)])
def test_split_tiles_match_oracle(gpu, batch, dtype, heads, kv_heads, head_dim):
    from vllm_rlt.kernels._hip import library

    lib = library()
    inputs = prefill_inputs(BATCHES[batch], heads, kv_heads, head_dim, dtype, gpu, seed=5)
    base, full = sizes(lib, inputs)
    assert full > base  # this call splits
    expected = oracle_prefill(*inputs[:6])
    # 0xFF bytes are NaN in fp32: a partial read before it is written shows.
    assert_close(call(lib, inputs, full), expected, dtype)
    # The smaller workspace of a caller that knows nothing of splits still works.
    assert_close(call(lib, inputs, base), expected, dtype)
    assert_close(call(lib, inputs, full - 1), expected, dtype)


@pytest.mark.parametrize("sequences,split", [
    ([(40, 40), (30, 30), (1300, 1), (17, 1)], False),  # wide tables, nothing to split
    ([(1200, 40), (30, 30), (90, 1), (17, 1)], True),
    ([(1300, 1), (20, 1), (3, 3), (60, 20)], False)])
@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim", [
    (torch.bfloat16, 8, 8, 128), (torch.float16, 6, 2, 64), (torch.bfloat16, 2, 1, 32)])
def test_decode_rows_merged_beside_the_tiles(gpu, sequences, split, dtype, heads, kv_heads,
                                             head_dim):
    """One launch merges the split decode rows and the tiles' key splits: the rows'
    bits are those of a call without key splits, and the tiles' too where no tile
    turns out to be split."""
    from vllm_rlt.kernels._hip import library

    lib = library()
    inputs = prefill_inputs(sequences, heads, kv_heads, head_dim, dtype, gpu, seed=11)
    base, full = sizes(lib, inputs)
    assert full > base
    merged, unsplit = call(lib, inputs, full), call(lib, inputs, base)
    assert_close(merged, oracle_prefill(*inputs[:6]), dtype)
    at = 0
    for _, queries in sequences:
        if queries == 1 or not split:
            assert torch.equal(merged[at : at + queries], unsplit[at : at + queries])
        at += queries


def test_split_prefill_in_a_graph_follows_the_device_lengths(gpu):
    """Captured once with wide tables, replayed after the lengths changed: the
    runs come from the device lengths, the grid only from the shapes."""
    from vllm_rlt.kernels.hip_attention import paged_prefill_attention

    sequences = [(1400, 100), (60, 30)]
    q, k, v, tables, lengths, cu, max_q = prefill_inputs(sequences, 8, 8, 128, torch.bfloat16,
                                                         gpu, seed=9)
    stream = torch.cuda.Stream()
    stream.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(stream):
        paged_prefill_attention(q, k, v, tables, lengths, cu, max_q)
    torch.cuda.current_stream().wait_stream(stream)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        captured = paged_prefill_attention(q, k, v, tables, lengths, cu, max_q)
    for n in (1400, 131, 100, 1024):
        lengths[0] = n
        captured.zero_()
        torch.cuda.synchronize()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(captured, paged_prefill_attention(q, k, v, tables, lengths, cu, max_q))
        assert_close(captured, oracle_prefill(q, k, v, tables, lengths, cu), torch.bfloat16)


@pytest.mark.parametrize("heads,kv_heads", [(2, 2), (8, 2), (16, 8)])
def test_longest_query_count_is_only_a_bound(gpu, heads, kv_heads):
    """max_seqlen_q up to INT32_MAX is accepted, whatever the group, and changes
    nothing: no sequence has more queries than the packed batch."""
    from vllm_rlt.kernels.hip_attention import paged_prefill_attention

    q, k, v, tables, lengths, cu, max_q = prefill_inputs([(300, 40), (77, 9)], heads, kv_heads, 64,
                                                         torch.bfloat16, gpu, seed=2)
    expected = paged_prefill_attention(q, k, v, tables, lengths, cu, max_q)
    assert_close(expected, oracle_prefill(q, k, v, tables, lengths, cu), torch.bfloat16)
    for bound in (q.shape[0], 2**31 - 1):
        assert torch.equal(paged_prefill_attention(q, k, v, tables, lengths, cu, bound), expected)


@pytest.mark.parametrize("dtype,offset,splits", [
    (torch.bfloat16, 0, True), (torch.float32, 0, False), (torch.bfloat16, 1, False)])
@pytest.mark.parametrize("plain", [True, False])
def test_only_calls_on_tiles_hold_room_for_splits(gpu, dtype, offset, splits, plain, monkeypatch):
    """A call that the tiles cannot take (float32, rows that are not 16-byte
    aligned) allocates no partials, through the extension module or ctypes."""
    from vllm_rlt.kernels import hip_attention

    if not plain:
        monkeypatch.setattr(hip_attention, "plain_calls", lambda: None)
    q, k, v, tables, lengths, cu, max_q = prefill_inputs([(1500, 100)], 8, 8, 64, dtype, gpu)
    shifted = torch.empty(q.numel() + offset, dtype=dtype, device=gpu)[offset:].view(q.shape)
    q = shifted.copy_(q)
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    out = hip_attention.paged_prefill_attention(q, k, v, tables, lengths, cu, max_q)
    peak = torch.cuda.max_memory_allocated() - before
    assert (peak > 1 << 20) == splits, peak  # the output and decode partials take 0.3 MiB
    assert_close(out, oracle_prefill(q, k, v, tables, lengths, cu), dtype)


@pytest.mark.parametrize("plain", [True, False])
def test_call_without_room_for_splits_runs_unsplit(gpu, plain, monkeypatch):
    """When the allocator cannot give the partials (a pool sized to the last of
    the memory), the call runs as with the smaller workspace, bit for bit."""
    from vllm_rlt.kernels import hip_attention
    from vllm_rlt.kernels._hip import library

    if not plain:
        monkeypatch.setattr(hip_attention, "plain_calls", lambda: None)
    inputs = prefill_inputs([(1500, 129)], 16, 16, 128, torch.bfloat16, gpu, seed=4)
    base, full = sizes(library(), inputs)
    assert full > base + (12 << 20)
    unsplit = call(library(), inputs, base)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(gpu).total_memory
    held = []
    try:
        # Room for the output (0.5 MiB) and the small workspace (0.2 MiB) only.
        torch.cuda.set_per_process_memory_fraction(
            (torch.cuda.memory_reserved() + (8 << 20)) / total)
        with pytest.raises(torch.OutOfMemoryError):
            while True:
                held.append(torch.empty(12 << 20, dtype=torch.uint8, device=gpu))
        out = hip_attention.paged_prefill_attention(*inputs)
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
        del held
    assert torch.equal(out, unsplit)
