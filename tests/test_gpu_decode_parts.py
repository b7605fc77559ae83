"""Decode splits cut into parts: a row's result must not depend on whether one
wave ran the parts one after another (launches with many splits) or a workgroup
ran them side by side (launches with few): torch.equal between a row alone and
the same row in a batch, and both against the oracle (tolerances of
test_gpu_attention). Sizes: splits of one part up to the most, a last part of one
page, pages that are no power of two, more than 64 pages to a part, a window that
starts inside a page; the MFMA kernel, and 1, 2, 4 and 8 heads a wave with 4, 8, 16
and 32 lanes to a token.
"""

import os
import re

import pytest
import torch

from conftest import PACKAGE_ROOT
from test_gpu_attention import assert_close, oracle_decode, random_paged

LENGTHS = [
    ((4097, 1025, 3000, 2049, 64), 16, 0),
    ((8193, 600, 8192), 16, 0),
    ((48000, 24001), 16, 0),
    ((5003, 77), 5, 0),                     # divided, not shifted
    ((9000, 1500), 1, 0),                   # more than 64 pages to a part
    ((6001, 5999), 16, 4501),               # window starting inside a page
]
# dtype, heads, kv_heads, head_dim, heads a wave (0: MFMA)
CONFIGS = [
    (torch.bfloat16, 2, 2, 128, 1), (torch.float16, 4, 1, 128, 4), (torch.bfloat16, 8, 1, 128, 0),
    (torch.float16, 16, 1, 64, 0), (torch.float32, 2, 1, 128, 1), (torch.bfloat16, 1, 1, 96, 1),
    (torch.bfloat16, 2, 2, 64, 1), (torch.bfloat16, 2, 2, 32, 1), (torch.bfloat16, 4, 2, 64, 2),
    (torch.bfloat16, 8, 1, 32, 8), (torch.float32, 8, 1, 64, 8)]


def constant(name):
    with open(os.path.join(PACKAGE_ROOT, "csrc", "paged_decode.hip")) as source:
        return int(re.search(rf"constexpr int {name} = (\d+);", source.read())[1])


def parts(n, block, window, dtype, head_dim, per_wave):
    """Parts of a row's full splits, as the kernel's partition has them."""
    size = 4 if dtype is torch.float32 else 2
    tokens = min(constant("kSplitTokens"), constant("kSplitBytes") // (head_dim * size))
    shortest = max(1, tokens // block)
    long = max(shortest, min(constant("kSplitTokens"), 2 * tokens) // block)
    start = max(0, n - window) if window else 0
    pages = -(-n // block) - start // block
    least = shortest if long < pages <= constant("kShortSplits") * shortest else long
    split = max(least, -(-pages // 16))
    if split <= 4 * shortest:
        return 1
    lanes = 1
    while lanes * 16 // size < head_dim:
        lanes *= 2
    chunk = 32 if per_wave == 0 else min(8, 16 // per_wave) * (64 // lanes)
    unit = max(1, chunk // block)
    most = constant("kParts" if per_wave == 1 else "kGroupParts")
    part = max(2 * shortest, -(-(-(-split // most)) // unit) * unit)
    return -(-split // part)


@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim,per_wave", CONFIGS)
def test_lengths_reach_every_number_of_parts(dtype, heads, kv_heads, head_dim, per_wave):
    """What the GPU test below is meant to cover, by the kernel's own constants."""
    counts = {parts(n, block, window, dtype, head_dim, per_wave)
              for lengths, block, window in LENGTHS for n in lengths}
    most = constant("kParts" if per_wave == 1 else "kGroupParts")
    assert {1, most} <= counts and len(counts) > 2 and max(counts) == most


@pytest.mark.gpu
@pytest.mark.parametrize("lengths,block,window", LENGTHS)
@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim,per_wave", CONFIGS)
def test_parts_side_by_side_equal_parts_in_turn(gpu, dtype, heads, kv_heads, head_dim, per_wave,
                                                lengths, block, window):
    from vllm_rlt.kernels.hip_attention import paged_attention

    q, k, v, tables, context = random_paged(list(lengths), heads, kv_heads, head_dim, dtype, gpu,
                                            block=block, seed=sum(lengths))
    # More workgroups than are resident at once: each row many times over.
    repeat = 1 + -(-3 * constant("kCus") // (16 * kv_heads) // len(lengths)) * 2
    index = torch.arange(len(lengths), device=gpu).repeat(repeat)
    many = paged_attention(q[index], k, v, tables[index].contiguous(), context[index], window)
    few = paged_attention(q, k, v, tables, context, window)
    expected = oracle_decode(q, k, v, tables, context, window)
    for row in range(len(lengths)):
        alone = paged_attention(q[row : row + 1], k, v, tables[row : row + 1].contiguous(),
                                context[row : row + 1], window)
        assert torch.equal(alone[0], few[row]), row
        assert torch.equal(alone[0], many[row]), row
        assert torch.equal(alone[0], many[len(lengths) * (repeat - 1) + row]), row
        assert_close(alone, expected[row : row + 1], dtype)


@pytest.mark.gpu
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
