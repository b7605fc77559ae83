"""Contexts close to what an int32 length can say: page and token arithmetic stays
in range. The pools are tiny (the tables repeat a few pages), so the expected
result is that of the distinct tokens alone.
"""

import pytest
import torch

from test_gpu_attention import assert_close, oracle_decode

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
