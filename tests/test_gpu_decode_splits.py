"""How rows are cut into splits: read back from which split partials a call writes
(the workspace is NaN before), for the fine splits of short rows, rows of a single
split and long rows; with tables just as wide as the row, where the launch has no
more split columns than the row needs, and wider ones. Every row is compared with
the oracle as well (tolerances of test_gpu_attention).
"""

import pytest
import torch

from test_gpu_attention import assert_close, oracle_decode, random_paged

pytestmark = pytest.mark.gpu


def splits_written(q, k, v, tables, lengths):
    """(output, number of split partials per row and head)."""
    from vllm_rlt.kernels._hip import library
    from vllm_rlt.kernels.hip_attention import dtype_code

    lib = library()
    rows, heads, dim = q.shape
    nbytes = lib.vrh_paged_decode_workspace_bytes(rows, heads, dim)
    workspace = torch.full((nbytes,), 0xFF, dtype=torch.uint8, device=q.device)
    out = torch.empty_like(q)
    lib.check(lib.vrh_paged_decode(
        dtype_code(q.dtype), out.data_ptr(), q.data_ptr(), k.data_ptr(), v.data_ptr(),
        tables.data_ptr(), lengths.data_ptr(), rows, heads, k.shape[2], dim, k.shape[1],
        tables.shape[1], tables.stride(0), q.stride(0), q.stride(1), out.stride(0), out.stride(1),
        *k.stride()[:3], *v.stride()[:3], 0, workspace.data_ptr(), nbytes,
        torch.cuda.current_stream().cuda_stream), "vrh_paged_decode")
    ml = workspace[: rows * heads * 16 * 2 * 4].view(torch.float32).view(rows, heads, 16, 2)
    return out, (~ml.isnan()).all(-1).sum(-1).cpu()


def expected_splits(n, short, block=16):
    """Splits of 2 * short tokens (at most 128), of ``short`` in rows of more than one
    such split and up to six short ones, 16 splits at most."""
    long = min(128, 2 * short)
    pages = -(-n // block)
    least = short if long // block < pages <= 6 * short // block else long
    count = -(-pages // max(least // block, -(-pages // 16)))
    return 0 if count == 1 else count  # a single split writes the output


@pytest.mark.parametrize("dtype,heads,kv_heads,head_dim,short", [
    (torch.bfloat16, 2, 2, 128, 64), (torch.float32, 2, 2, 128, 32), (torch.float16, 2, 2, 64, 128),
    (torch.float16, 4, 1, 128, 128), (torch.bfloat16, 8, 1, 128, 128),  # grouped: no short ones
    (torch.float32, 8, 1, 128, 128)])
@pytest.mark.parametrize("wider", [0, 200])
def test_splits_follow_the_row_length(gpu, dtype, heads, kv_heads, head_dim, short, wider):
    long = min(128, 2 * short)
    for n in (1, short, short + 1, long, long + 1, 3 * short + 5, 6 * short, 6 * short + 1,
              8 * long + 1, 16 * long, 16 * long + 1, 5000):
        q, k, v, tables, lengths = random_paged([n], heads, kv_heads, head_dim, dtype, gpu, seed=n)
        tables = torch.nn.functional.pad(tables, (0, wider), value=-1)
        out, written = splits_written(q, k, v, tables, lengths)
        assert (written == expected_splits(n, short)).all(), n
        assert_close(out, oracle_decode(q, k, v, tables, lengths), dtype)
