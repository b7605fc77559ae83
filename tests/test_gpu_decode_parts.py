"""Decode splits cut into parts: a row's result must not depend on whether one
wave ran the parts one after another (launches with many splits) or a workgroup
ran them side by side (launches with few): torch.equal between a row alone and
the same row in a batch, and both against the oracle (tolerances of
test_gpu_attention). Sizes: splits of one, two and the most parts, a last part
of one token, pages that are no power of two, more than 64 pages to a part, a
window that starts inside a page, both kernels and every lane width.
"""

import pytest
import torch

from test_gpu_attention import assert_close, oracle_decode, random_paged

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("lengths,block,window", [
    ((4097, 1025, 3000, 2049, 64), 16, 0),  # 2 to 5 parts a split, one whole split
    ((8193, 600, 8192), 16, 0),             # 8 parts, and a ninth page
    ((5003, 77), 5, 0),                     # divided, not shifted
    ((9000, 1500), 1, 0),                   # more than 64 pages to a part
    ((6001, 5999), 16, 4501),               # window starting inside a page
])
@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim", [
    (torch.bfloat16, 2, 2, 128), (torch.float16, 4, 1, 128), (torch.bfloat16, 8, 1, 128),
    (torch.float16, 16, 1, 64), (torch.float32, 2, 1, 128), (torch.bfloat16, 1, 1, 96)])
def test_parts_side_by_side_equal_parts_in_turn(gpu, dtype, heads, kv_heads, head_dim, lengths,
                                                block, window):
    from vllm_rlt.kernels.hip_attention import paged_attention

    q, k, v, tables, context = random_paged(list(lengths), heads, kv_heads, head_dim, dtype, gpu,
                                            block=block, seed=sum(lengths))
    # Over 1024 splits in one launch: each row many times over.
    repeat = 1 + 1024 // (16 * kv_heads) // len(lengths) * 2
    index = torch.arange(len(lengths), device=gpu).repeat(repeat)
    many = paged_attention(q[index], k, v, tables[index].contiguous(), context[index], window)
    expected = oracle_decode(q, k, v, tables, context, window)
    for row in range(len(lengths)):
        alone = paged_attention(q[row : row + 1], k, v, tables[row : row + 1].contiguous(),
                                context[row : row + 1], window)
        assert torch.equal(alone[0], many[row]), row
        assert torch.equal(alone[0], many[len(lengths) * (repeat - 1) + row]), row
        assert_close(alone, expected[row : row + 1], dtype)


def test_f16_pair_products_keep_small_values(gpu):
    """q.k on packed f16 pairs: subnormal f16 keys and queries count in full (the
    products are exact in fp32), as in the oracle."""
    from vllm_rlt.kernels.hip_attention import paged_attention

    q, k, v, tables, context = random_paged([200, 33], 2, 2, 128, torch.float16, gpu, seed=3)
    q = (q.float() * (6e4 / float(q.abs().max()))).to(torch.float16)
    k = (k.float() * 1.5e-5).clamp(-6e-5, 6e-5).to(torch.float16)  # subnormal
    assert float(k.abs().max()) < 6.2e-5 and float(k.abs().max()) > 0
    out = paged_attention(q, k, v, tables, context)
    assert_close(out, oracle_decode(q, k, v, tables, context), torch.float16)
    spread = oracle_decode(q, k * 0, v, tables, context)
    # The keys matter: ten times the tolerance.
    assert float((out.float().cpu() - spread.float()).abs().max()) > 0.02
