"""Contexts close to what an int32 length can say: page and token arithmetic stays
in range. The pools are tiny (the tables repeat a few pages), so the expected
result is that of the distinct tokens alone.
"""

import pytest
import torch

from test_gpu_attention import assert_close, oracle_decode, oracle_prefill

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype,heads,kv_heads", [
    (torch.bfloat16, 1, 1),      # a workgroup per split, one wave a part
    (torch.bfloat16, 64, 64),    # over 512 splits: parts one after another
    (torch.float32, 64, 64),
    (torch.bfloat16, 8, 1),      # the same for grouped-query heads on MFMA
    (torch.bfloat16, 528, 66)])  # (over 1024 splits)
def test_last_part_ends_with_the_row(gpu, dtype, heads, kv_heads):
    """626 pages of 128 tokens are visible: splits of 40 pages, the last one of 26,
    which is no whole number of parts (5 pages; 10 on MFMA). Four pages past the
    last token would be past 2^31."""
    from vllm_rlt.kernels.hip_attention import paged_attention

    block, pages = 128, 2**24 - 2
    gen = torch.Generator().manual_seed(heads)
    q, k, v = (torch.randn(*shape, generator=gen).to(dtype).to(gpu) for shape in
               [(1, heads, 128)] + 2 * [(2, block, kv_heads, 128)])
    tables = (torch.arange(pages, device=gpu) % 2).to(torch.int32).view(1, pages)
    lengths = torch.tensor([pages * block], dtype=torch.int32, device=gpu)
    out = paged_attention(q, k, v, tables, lengths, 626 * block)
    # Each of the two pages' tokens is seen 313 times.
    expected = oracle_decode(q, k, v, tables[:, :2], torch.tensor([2 * block]))
    assert_close(out, expected, dtype)


def test_unsplit_prefill_reads_every_key_of_a_very_long_context(gpu):
    """A tile that is not split along its keys covers the whole context: here 16
    queries over 2^29 keys and more, of which all but the last two pages weigh
    nothing (scores 85 lower), so the result is attention over those pages. One
    workgroup takes 2^24 steps: several seconds."""
    from vllm_rlt.kernels.hip_attention import dtype_code
    from vllm_rlt.kernels._hip import library

    lib = library()
    block, heads, dim, queries, far = 128, 1, 32, 16, 2**22
    gen = torch.Generator().manual_seed(7)
    q, k, v = (torch.randn(*shape, generator=gen) for shape in
               [(queries, heads, dim)] + 2 * [(3, block, heads, dim)])
    q[..., 0] = 8
    k[0, ..., 0], k[1:, ..., 0] = -60, 0
    q, k, v = (t.to(torch.bfloat16).to(gpu) for t in (q, k, v))
    tables = torch.zeros(1, far + 2, dtype=torch.int32, device=gpu)
    tables[0, far:] = torch.tensor([1, 2], dtype=torch.int32)
    lengths = torch.tensor([(far + 2) * block], dtype=torch.int32, device=gpu)
    cu = torch.tensor([0, queries], dtype=torch.int32, device=gpu)
    # The workspace without room for key splits.
    nbytes = lib.vrh_paged_prefill_workspace_bytes(1, queries, heads, dim)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=gpu)
    out = torch.empty_like(q)
    lib.check(lib.vrh_paged_prefill(
        dtype_code(q.dtype), out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        tables.data_ptr(), lengths.data_ptr(), cu.data_ptr(), 1, queries, queries, heads, heads,
        dim, block, tables.shape[1], tables.stride(0), q.stride(0), q.stride(1), out.stride(0),
        out.stride(1), *k.stride()[:3], *v.stride()[:3], workspace.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream), "vrh_paged_prefill")
    expected = oracle_prefill(q, k, v, tables[:, far:], torch.tensor([2 * block]), cu)
    assert_close(out, expected, q.dtype)
