"""Performance cases of the paged-KV path: what a serving program has it do, layer by layer.

Four kinds of call, each through the public entry point that a model runner uses:

  decode   ``create_backend("hip", ...)`` called with one query per row (``windowed`` with a window)
  prefill  its ``prefill``: packed causal chunks, one-query decode rows among them
  append   ``kv_append``: a step's new K/V rows into the pages of one layer
  silu     ``silu_and_mul``: the MLP activation beside attention

``listed()`` names twelve of them, ``draw(rng)`` gives others of the same ranges: 1 to 128 rows, contexts of 16
to 32768 tokens, 1 to 16 prompt chunks of 1 to 512 queries, appends of 1 to 8192 rows, activations of 1 to 8192
rows; bf16 mostly, f16 and f32 as well; 16 x 128 heads (multi-head) and 8 KV heads shared by 32 or 64 query
heads; pages of 16 tokens scattered over the pool. Lengths belong to the case (``lengths`` seeds them); values and
page placement come from the seed of ``prepare``.
"""

import math
import os
import random
import sys

import torch

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "vllm-rlt_amd"))

from vllm_rlt.attention import create_backend  # noqa: E402
from vllm_rlt.kernels.activation import silu_and_mul  # noqa: E402
from vllm_rlt.kernels.hip_attention import kv_append  # noqa: E402

BLOCK = 16
DTYPES = {"bf16": torch.bfloat16, "f16": torch.float16, "f32": torch.float32}
BYTES = {"bf16": 2, "f16": 2, "f32": 4}


def _decode(name=None, **kw):
    case = {"kind": "decode", "dtype": "bf16", "q_heads": 16, "kv_heads": 16, "head_dim": 128, "layers": 1,
            "rows": 1, "low": 16, "high": 512, "share": 1, "prefix": 0, "window": 0, "width": 0, "lengths": 2}
    case.update(kw)
    return {"name": name, **case} if name else case


def _prefill(name=None, **kw):
    case = {"kind": "prefill", "dtype": "bf16", "q_heads": 16, "kv_heads": 16, "head_dim": 128,
            "prompts": 1, "q_low": 512, "q_high": 512, "prefix_low": 0, "prefix_high": 0,
            "decode_rows": 0, "low": 256, "high": 4096, "lengths": 2}
    case.update(kw)
    return {"name": name, **case} if name else case


def listed():
    return [
        # One user's chat deep into a long context: a single row, latency of one token.
        _decode("decode_one_row_long", rows=1, low=24001, high=24001),
        # The fp32 check-out shape: 8 rows, short contexts, float32 pool.
        _decode("decode_fp32_8_rows", dtype="f32", rows=8, low=64, high=512),
        # The headline step: 64 requests, 16 x 128 heads, a pool of several layers.
        _decode("decode_64_rows", rows=64, layers=4, low=512, high=4096),
        # Grouped-query heads in float16, a batch that is no power of two.
        _decode("decode_gqa_f16", dtype="f16", q_heads=32, kv_heads=8, rows=37, low=300, high=6000),
        # Parallel samples of 16 prompts: 8 rows share a 1024-token prefix, private tails.
        _decode("decode_shared_prefix", rows=128, share=8, prefix=1024, low=64, high=1024),
        # Sliding-window attention under the fixed-width tables of a captured graph.
        _decode("decode_window_wide_table", rows=24, low=64, high=8192, window=1024, width=2048),
        # Long-context serving: many rows, up to 32768 tokens each.
        _decode("decode_long_batch", rows=96, low=2048, high=32768),
        # One request's prompt chunk with nothing else to run: time to first token.
        _prefill("prefill_one_chunk", prompts=1, prefix_low=6656, prefix_high=6656),
        # The mixed step: 16 prompts' chunks packed with 48 decode rows.
        _prefill("prefill_mixed", prompts=16, q_low=212, q_high=512, prefix_low=0, prefix_high=7680, decode_rows=48),
        # Short ragged prompts over grouped-query heads in float16, head_dim 64.
        _prefill("prefill_gqa_ragged_f16", dtype="f16", q_heads=32, kv_heads=8, head_dim=64, prompts=7, q_low=17,
                 q_high=390, prefix_low=0, prefix_high=2900),
        # The mixed step's K/V written into the pages of one layer.
        {"name": "append_chunks", "kind": "append", "dtype": "bf16", "kv_heads": 16, "head_dim": 128, "rows": 8039, "run": 512},
        # The MLP activation of the same step.
        {"name": "silu_prefill", "kind": "silu", "dtype": "bf16", "rows": 8192, "width": 5632, "offset": 0},
    ]


def _log(rng, low, high):
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["decode"] * 5 + ["prefill"] * 3 + ["append", "silu"])
    seed = rng.randrange(1 << 20)
    if kind == "append":
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "f16", "f32"]), "kv_heads": rng.choice([8, 16]),
                "head_dim": rng.choice([64, 128]), "rows": _log(rng, 1, 8192), "run": _log(rng, 1, 512)}
    if kind == "silu":
        dtype = rng.choice(["bf16", "bf16", "f16", "f32"])
        return {"kind": kind, "dtype": dtype, "rows": _log(rng, 1, 8192 if dtype != "f32" else 4096),
                "width": rng.choice([2048, 5632, 5632, 5633]), "offset": rng.choice([0, 0, 0, 1])}
    q_heads, kv_heads = rng.choice([(16, 16), (16, 16), (32, 8), (64, 8)])
    heads = {"q_heads": q_heads, "kv_heads": kv_heads, "lengths": seed}
    if kind == "prefill":
        high = _log(rng, 16, 512)
        prefix = rng.choice([0, _log(rng, 16, 7680)])
        prompts = _log(rng, 1, 16 if q_heads == 16 else 8 if q_heads == 32 else 4)
        return _prefill(dtype=rng.choice(["bf16", "bf16", "f16"]), head_dim=rng.choice([64, 128, 128]), prompts=prompts,
                        q_low=rng.randint(1, high), q_high=high, prefix_low=rng.randint(0, prefix), prefix_high=prefix,
                        decode_rows=rng.choice([0, _log(rng, 1, 48)]), **heads)
    dtype = rng.choice(["bf16", "bf16", "bf16", "f16", "f32"])
    rows = _log(rng, 1, 128)
    # No more K/V than the longest listed batch reads (float32 tokens are twice as long).
    top = min(32768, 96 * 15000 * 2 * 16 * 128 // (rows * kv_heads * 128 * BYTES[dtype] // 2))
    high = _log(rng, 64, top)
    share = rng.choice([1, 1, 1, 4])
    return _decode(dtype=dtype, head_dim=rng.choice([64, 128, 128]), rows=rows, low=rng.randint(16, high), high=high,
                   share=share, prefix=0 if share == 1 else min(1024, high // 2) // BLOCK * BLOCK,
                   window=rng.choice([0, 0, 0, _log(rng, 128, 2048)]), width=rng.choice([0, 0, 2048 + 64]), **heads)


def _spread(seed, count, low, high):
    rng = random.Random(seed)
    return [rng.randint(low, high) for _ in range(count)]


def _decode_lengths(case):
    return [case["prefix"] + n for n in _spread(case["lengths"], case["rows"], case["low"], case["high"])]


def _sequences(case):
    """(query count, context length) of every sequence of a packed batch: the chunks, then the decode rows."""
    qs = _spread(case["lengths"], case["prompts"], case["q_low"], case["q_high"])
    before = _spread(case["lengths"] + 1, case["prompts"], case["prefix_low"], case["prefix_high"])
    rows = _spread(case["lengths"] + 2, case["decode_rows"], case["low"], case["high"])
    return [(q, p + q) for q, p in zip(qs, before)] + [(1, n) for n in rows]


def _pages(n):
    return -(-n // BLOCK)


def _tables(counts, width, gen, device, share=1, prefix=0):
    """Tables over one scattered pool, -1 padded; rows of a group of ``share`` alias the group's prefix pages."""
    lead = prefix // BLOCK
    groups = -(-len(counts) // share) if lead else 0
    total = groups * lead + sum(c - lead for c in counts)
    order = torch.randperm(total, generator=gen, device=device).to(torch.int32)
    tables = torch.full((len(counts), max(width, max(counts))), -1, dtype=torch.int32, device=device)
    at = groups * lead
    for r, count in enumerate(counts):
        if lead:
            tables[r, :lead] = order[r // share * lead : (r // share + 1) * lead]
        tables[r, lead:count] = order[at : at + count - lead]
        at += count - lead
    return tables, total


def _pool(case, blocks, layers, gen, device):
    shape = (blocks, layers, BLOCK, case["kv_heads"], case["head_dim"])
    return [torch.empty(shape, dtype=DTYPES[case["dtype"]], device=device).normal_(generator=gen) for _ in range(2)]


def prepare(case, seed):
    device = torch.device("cuda")
    gen = torch.Generator(device=device).manual_seed(seed)
    dtype = DTYPES[case["dtype"]]
    kind = case["kind"]

    def values(*shape):
        return torch.empty(shape, dtype=dtype, device=device).normal_(generator=gen)

    if kind == "silu":
        count, skip = case["rows"] * case["width"], case["offset"]
        gate, up = (values(count + skip)[skip:].view(case["rows"], case["width"]) for _ in range(2))
        return {"kind": kind, "gate": gate, "up": up}
    if kind == "append":
        rows = case["rows"]
        runs = -(-rows // case["run"])
        per = _pages(case["run"] + BLOCK - 1)  # a run starts anywhere in its first page
        blocks = 2 * runs * per
        pages = torch.randperm(blocks, generator=gen, device=device)[: runs * per].view(runs, per)
        start = torch.randint(0, BLOCK, (runs, 1), generator=gen, device=device)
        pos = start + torch.arange(case["run"], device=device)
        k_cache, v_cache = _pool(case, blocks, 1, gen, device)
        shape = (rows, case["kv_heads"], case["head_dim"])
        return {"kind": kind, "k_cache": k_cache[:, 0], "v_cache": v_cache[:, 0], "k": values(*shape), "v": values(*shape),
                "blocks": pages.gather(1, pos // BLOCK).reshape(-1)[:rows].contiguous(),
                "offsets": (pos % BLOCK).reshape(-1)[:rows].contiguous()}
    backend = create_backend("hip", device, dtype, case["head_dim"], BLOCK)
    if kind == "prefill":
        seqs = _sequences(case)
        lengths = [n for _, n in seqs]
        tables, blocks = _tables([_pages(n) for n in lengths], 0, gen, device)
        k_cache, v_cache = _pool(case, blocks, 1, gen, device)
        cu = [0]
        for q, _ in seqs:
            cu.append(cu[-1] + q)
        return {"kind": kind, "backend": backend, "q": values(cu[-1], case["q_heads"], case["head_dim"]),
                "k_cache": k_cache[:, 0], "v_cache": v_cache[:, 0], "tables": tables,
                "lengths": torch.tensor(lengths, dtype=torch.int32, device=device),
                "cu": torch.tensor(cu, dtype=torch.int32, device=device), "max_q": max(q for q, _ in seqs)}
    lengths = _decode_lengths(case)
    tables, blocks = _tables([_pages(n) for n in lengths], case["width"], gen, device, case["share"], case["prefix"])
    k_cache, v_cache = _pool(case, blocks, case["layers"], gen, device)
    layer = case["layers"] // 2
    return {"kind": kind, "backend": backend, "q": values(case["rows"], case["q_heads"], case["head_dim"]),
            "k_cache": k_cache[:, layer], "v_cache": v_cache[:, layer], "tables": tables,
            "lengths": torch.tensor(lengths, dtype=torch.int32, device=device), "window": case["window"]}


def run(state):
    s = state
    if s["kind"] == "decode":
        if s["window"]:
            return s["backend"].windowed(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["lengths"], s["window"])
        return s["backend"](s["q"], s["k_cache"], s["v_cache"], s["tables"], s["lengths"])
    if s["kind"] == "prefill":
        return s["backend"].prefill(s["q"], s["k_cache"], s["v_cache"], s["tables"], s["lengths"], s["cu"], s["max_q"])
    if s["kind"] == "append":
        kv_append(s["k_cache"], s["v_cache"], s["k"], s["v"], s["blocks"], s["offsets"])
        return s["k_cache"], s["v_cache"]
    return silu_and_mul(s["gate"], s["up"])


def work(case):
    es = BYTES[case["dtype"]]
    if case["kind"] == "silu":
        count = case["rows"] * case["width"]
        return {"bytes": 3 * count * es, "flops": 5 * count}
    if case["kind"] == "append":
        return {"bytes": case["rows"] * (4 * case["kv_heads"] * case["head_dim"] * es + 16), "flops": 0}
    token = 2 * case["kv_heads"] * case["head_dim"] * es
    query = case["q_heads"] * case["head_dim"]
    if case["kind"] == "prefill":
        seqs = _sequences(case)
        pairs = sum(q * n - q * (q - 1) // 2 for q, n in seqs)
        return {"bytes": sum(n * token + 2 * q * query * es + 4 * _pages(n) for q, n in seqs), "flops": 4 * query * pairs}
    total = read = 0
    for r, n in enumerate(_decode_lengths(case)):
        seen = min(n, case["window"]) if case["window"] else n
        total += seen
        # A group's shared prefix is read once for all of its rows.
        aliased = max(0, case["prefix"] - (n - seen)) if r % case["share"] else 0
        read += (seen - aliased) * token + 4 * _pages(seen) + 2 * query * es
    return {"bytes": read, "flops": 4 * query * total}


def tolerance(case):
    if case["kind"] in ("append", "silu"):
        return "exact"  # byte copies; SiLU rounds like the double expression, bit for bit
    return {"bf16": {"rel": 1e-2, "max": 8e-2}, "f16": {"rel": 1.5e-3, "max": 1.2e-2}, "f32": {"rel": 1e-5, "max": 1e-4}}[case["dtype"]]


def _attend(q, k, v, first, start):
    """Softmax attention in float64: q [n, Hq, D] at positions first.., k and v [m, Hkv, D] at positions start.. ."""
    n, heads, dim = q.shape
    kv = k.shape[1]
    group = heads // kv
    qd = q.double().view(n, kv, group, dim).permute(1, 2, 0, 3).reshape(kv, group * n, dim).contiguous()
    kd, vd = k.double().permute(1, 2, 0).contiguous(), v.double().permute(1, 0, 2).contiguous()
    scores = torch.matmul(qd, kd).view(kv, group, n, -1) / math.sqrt(dim)
    if n > 1:
        pos = torch.arange(k.shape[0], device=q.device) + start
        scores.masked_fill_(pos[None, :] > first + torch.arange(n, device=q.device)[:, None], -math.inf)
    out = torch.matmul(torch.softmax(scores, -1).view(kv, group * n, -1), vd)
    return out.view(kv, group, n, dim).permute(2, 0, 1, 3).reshape(n, heads, dim)


def exact(case, seed):
    s = prepare(case, seed)
    if case["kind"] == "silu":
        gate = s["gate"].double()
        # The activation is defined with SiLU rounded to the storage type before the product.
        return (gate * torch.sigmoid(gate)).to(s["gate"].dtype).double() * s["up"].double()
    if case["kind"] == "append":
        for cache, new in ((s["k_cache"], s["k"]), (s["v_cache"], s["v"])):
            cache[s["blocks"], s["offsets"]] = new
        return s["k_cache"].double(), s["v_cache"].double()

    def context(row, start, end):
        pages = s["tables"][row, start // BLOCK : _pages(end)].long()
        cut = slice(start % BLOCK, start % BLOCK + end - start)
        return [c[pages].flatten(0, 1)[cut] for c in (s["k_cache"], s["v_cache"])]

    out = torch.empty(s["q"].shape, dtype=torch.float64, device=s["q"].device)
    if case["kind"] == "prefill":
        at = 0
        for row, (q, n) in enumerate(_sequences(case)):
            out[at : at + q] = _attend(s["q"][at : at + q], *context(row, 0, n), n - q, 0)
            at += q
        return out
    for row, n in enumerate(_decode_lengths(case)):
        start = max(0, n - case["window"]) if case["window"] else 0
        out[row : row + 1] = _attend(s["q"][row : row + 1], *context(row, start, n), n - 1, start)
    return out
