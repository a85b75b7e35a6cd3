"""Segments launched together give each segment's own bits.

HBM-resident runs launch up to 32 segments at once, ordered by their keys;
each must get the output and LSE of a run that has it alone: empty, one-row
and ragged segments, more than one launch's worth, heads that are and are not
a multiple of the XCDs, causal with queries that see no key.
"""

from __future__ import annotations

import ctypes
import itertools
import random

import pytest
import torch

from seqattn import StreamingAttentionConfig, StreamingAttentionRunner, build_plan, _native

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim,dtype,count", [
    (8, 2, 128, torch.bfloat16, 40),
    (16, 16, 64, torch.float16, 33),
    (6, 3, 96, torch.bfloat16, 32),
    (8, 8, 256, torch.bfloat16, 2),
    (4, 1, 32, torch.float16, 5),
])
def test_segments_together_equal_each_alone(q_heads, kv_heads, head_dim, dtype, count, causal):
    print(f"[gpu case] segments {count} heads={q_heads}/{kv_heads} d={head_dim} {dtype} causal={causal}", flush=True)
    rng = random.Random(count)
    q_lengths = [rng.choice([0, 1, 17, 128, 129, 300]) for _ in range(count)]
    k_lengths = [n and rng.choice([1, 63, 64, 65, 200, 700]) for n in q_lengths]
    q_lengths[0], k_lengths[0] = 400, 650
    cu_q, cu_k = ([0, *itertools.accumulate(x)] for x in (q_lengths, k_lengths))
    gen = torch.Generator(device="cuda").manual_seed(7)
    q, k, v = (torch.randn((n, h, head_dim), generator=gen, device="cuda").to(dtype)
               for n, h in ((cu_q[-1], q_heads), (cu_k[-1], kv_heads), (cu_k[-1], kv_heads)))
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=256, kv_chunk_tokens=192)
    plan = build_plan(q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, dtype=dtype, device="cuda",
                      max_q_tokens=cu_q[-1], max_kv_tokens=cu_k[-1], config=config)
    runner = StreamingAttentionRunner(plan, config)
    out, lse = runner(q, k, v, torch.tensor(cu_q), torch.tensor(cu_k), causal=causal, return_lse=True)
    for s in range(count):
        rows, keys = slice(cu_q[s], cu_q[s + 1]), slice(cu_k[s], cu_k[s + 1])
        if q_lengths[s] == 0:
            continue
        alone, alone_lse = runner(q[rows], k[keys], v[keys], torch.tensor([0, q_lengths[s]]),
                                  torch.tensor([0, k_lengths[s]]), causal=causal, return_lse=True)
        assert torch.equal(out[rows], alone), s
        assert torch.equal(lse[:, rows], alone_lse), s
    torch.cuda.synchronize()
    runner.close()


def test_broadcast_v_rows_are_read_through_the_transposed_copy():
    """V with a token stride of 0 cannot be read in place: it takes the copy whatever the segment's size."""
    print("[gpu case] segments V token stride 0", flush=True)
    heads, kv_heads, n, d = 8, 2, 200, 128
    gen = torch.Generator(device="cuda").manual_seed(3)
    q, k, v = (torch.randn((t, h, d), generator=gen, device="cuda").to(torch.bfloat16)
               for t, h in ((n, heads), (n, kv_heads), (1, kv_heads)))
    bounds = (ctypes.c_int64 * 3)(0, 77, n)

    def run(values):
        out, lse = torch.empty_like(q), torch.empty((heads, n), device="cuda")
        _native.check(_native.lib().sa_run_resident_noalloc(
            q.data_ptr(), k.data_ptr(), values.data_ptr(), out.data_ptr(), lse.data_ptr(), *q.stride()[:2],
            *k.stride()[:2], *values.stride()[:2], *out.stride()[:2], lse.stride(0), bounds, bounds, 2, heads, kv_heads,
            d, _native.SA_DTYPE_BF16, 128, 0.09, 1, torch.cuda.current_stream().cuda_stream), "sa_run_resident_noalloc")
        return out, lse

    broadcast = v.expand(n, kv_heads, d)
    assert broadcast.stride(0) == 0
    results = run(broadcast), run(broadcast.contiguous())
    torch.cuda.synchronize()
    for a, b in zip(*results):
        assert torch.equal(a, b)


@pytest.mark.parametrize("rows,count", [(1_200_000_000, 1), (34_000_000, 34)])
def test_more_queries_than_one_launch_holds(rows, count):
    """2.4e9 and 2.3e9 query x head pairs at head_dim 16: more than a launch's
    2^32 threads, in one segment and over segments.  Every query is the same
    row (token stride 0), so every output row is that of a small run."""
    print(f"[gpu case] segments of {rows} x {count} queries", flush=True)
    heads, d, keys = 2, 16, 64
    gen = torch.Generator(device="cuda").manual_seed(5)
    q, k, v = (torch.randn((n, heads, d), generator=gen, device="cuda").to(torch.bfloat16) for n in (1, keys, keys))
    config = StreamingAttentionConfig(kv_chunk_tokens=64)
    plan = build_plan(q_heads=heads, kv_heads=heads, head_dim=d, dtype=torch.bfloat16, device="cuda", max_q_tokens=256,
                      max_kv_tokens=keys * count, config=config)
    runner = StreamingAttentionRunner(plan, config)
    expected = runner(q, k, v, torch.tensor([0, 1]), torch.tensor([0, keys]))
    total = rows * count
    out = torch.empty((total, heads, d), dtype=torch.bfloat16, device="cuda")
    k_all, v_all = (x.repeat(count, 1, 1) for x in (k, v))
    cu_q, cu_k = ((ctypes.c_int64 * (count + 1))(*range(0, n * count + 1, n)) for n in (rows, keys))
    workspace = runner._workspace
    _native.check(_native.lib().sa_pipeline_run_resident(
        workspace.handle, q.data_ptr(), k_all.data_ptr(), v_all.data_ptr(), out.data_ptr(), None, 0, d, heads * d, d,
        heads * d, d, heads * d, d, 0, cu_q, cu_k, count, d**-0.5, 0, workspace.compute_stream.cuda_stream, None),
        "sa_pipeline_run_resident")
    step = 50_000_000
    for start in range(0, total, step):
        assert bool((out[start:start + step] == expected).all()), start
    torch.cuda.synchronize()
    runner.close()
    del out
    torch.cuda.empty_cache()  # 70 GB and more
