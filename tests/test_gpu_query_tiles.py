"""The update kernel's workgroup widths (128, 256 and 384 queries) and LDS stages give the same bits.

A launch picks its width and stages for speed; a query's online softmax must
not depend on which other queries share its workgroup, nor on how many tiles
are in flight.  Each launch below asserts the shape it takes.
"""

from __future__ import annotations

import ctypes
import itertools

import pytest
import torch

from seqattn import StreamingAttentionConfig, StreamingAttentionRunner, StreamingAttentionStats, _native, build_plan
from seqattn.kernels import update_attention_state, update_attention_state_int8

pytestmark = pytest.mark.gpu

ROWS, TRANSPOSED_V, INT8 = range(3)  # kv_layout


def launch_shape(q_tokens, kv_tokens, heads, head_dim, *, causal, causal_shift=0, kv_layout=ROWS):
    """(rows of a workgroup, LDS stages) of the launch over these segments."""
    arrays = [(ctypes.c_int32 * len(x))(*x) for x in (q_tokens, kv_tokens)]
    rows, stages, workgroups = ctypes.c_int32(), ctypes.c_int32(), ctypes.c_int64()
    _native.check(_native.lib().sa_update_launch_shape(
        *arrays, len(q_tokens), *heads, head_dim, causal_shift, int(causal), kv_layout, 0, rows, stages, workgroups),
        "sa_update_launch_shape")
    return rows.value, stages.value


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("head_dim,rows,int8,width", [
    (16, 2000, False, 256), (32, 2000, False, 256), (32, 1000, True, 256), (64, 2000, False, 256),
    (64, 1000, True, 256), (96, 1000, False, 256), (96, 1500, False, 384), (128, 1000, False, 256),
    (128, 1500, False, 384), (128, 1000, True, 256), (128, 1500, True, 384), (256, 1000, False, 256),
])
def test_workgroup_widths_give_the_same_state(head_dim, rows, int8, width, causal, dtype):
    """The wide workgroups against slices of 100 queries, which take the narrow ones."""
    print(f"[gpu case] widths d={head_dim} rows={rows} int8={int8} causal={causal} {dtype}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    heads, kv_heads, keys = 64, 8, rows + 1530
    q = torch.randn((rows, heads, head_dim), generator=gen, device="cuda").to(dtype)
    if int8:
        k, v = (torch.randint(-127, 128, (keys, kv_heads, head_dim), generator=gen, device="cuda", dtype=torch.int8)
                for _ in range(2))
        scales = [torch.rand((-(-keys // 64), kv_heads), generator=gen, device="cuda").mul_(0.05).half()
                  for _ in range(2)]
    else:
        k, v = (torch.randn((keys, kv_heads, head_dim), generator=gen, device="cuda").to(dtype)
                for _ in range(2))

    layout = INT8 if int8 else ROWS
    assert launch_shape([rows], [keys], (heads, kv_heads), head_dim, causal=causal, causal_shift=keys - rows,
                        kv_layout=layout)[0] == width

    def run(start, stop, m, l, acc):
        if stop - start < rows:
            assert launch_shape([stop - start], [keys], (heads, kv_heads), head_dim, causal=causal,
                                causal_shift=start + keys - rows, kv_layout=layout)[0] == 128
        common = dict(q_tokens=stop - start, kv_tokens=keys, q_local_offset=start, kv_local_offset=0,
                      causal_shift=keys - rows, softmax_scale=head_dim**-0.5, causal=causal, initialize=True)
        if int8:
            update_attention_state_int8(q[start:stop], k, v, *scales, m, l, acc, storage_token_offset=0, **common)
        else:
            update_attention_state(q[start:stop], k, v, m, l, acc, **common)

    def state():
        return (torch.empty((rows, heads), device="cuda"), torch.empty((rows, heads), device="cuda"),
                torch.empty((rows, heads, head_dim), device="cuda"))

    whole, sliced = state(), state()
    run(0, rows, *whole)
    for start in range(0, rows, 100):
        stop = min(start + 100, rows)
        run(start, stop, *(t[start:stop] for t in sliced))
    torch.cuda.synchronize()
    for name, a, b in zip(("running_max", "running_sum", "accumulator"), whole, sliced):
        assert torch.isfinite(a).all(), name
        assert torch.equal(a, b), name


@pytest.mark.parametrize("head_dim,dtype", [(32, torch.bfloat16), (64, torch.float16), (80, torch.bfloat16),
                                            (128, torch.float16)])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("tail", [0, 1, 63, 65, 130])
def test_small_launches_over_many_keys_keep_more_tiles_in_flight_and_give_the_same_state(head_dim, dtype, causal, tail):
    """300 heads are more workgroups than CUs (two LDS stages); 150 of them are fewer (four, over 32 MB of K and V)."""
    print(f"[gpu case] stages d={head_dim} causal={causal} tail={tail}", flush=True)
    heads, part, rows = 300, 150, 3
    keys = max(1024, -(-(33 << 20) // (4 * part * head_dim)) // 64 * 64 + 64) + tail
    for n, stages in ((heads, 2), (part, 4)):
        assert launch_shape([rows], [keys], (n, n), head_dim, causal=causal, causal_shift=keys - rows - 40) == (128, stages)
    gen = torch.Generator(device="cuda").manual_seed(11)
    q, k, v = (torch.randn((n, heads, head_dim), generator=gen, device="cuda").to(dtype) for n in (rows, keys, keys))

    def run(heads_of):
        n = q[:, heads_of].shape[1]
        state = (torch.empty((rows, n), device="cuda"), torch.empty((rows, n), device="cuda"),
                 torch.empty((rows, n, head_dim), device="cuda"))
        for initialize in (True, False):  # a new state, then one that is loaded
            update_attention_state(q[:, heads_of], k[:, heads_of], v[:, heads_of], *state, q_tokens=rows,
                                   kv_tokens=keys, q_local_offset=0, kv_local_offset=0, causal_shift=keys - rows - 40,
                                   softmax_scale=0.1, causal=causal, initialize=initialize)
        return state

    whole = run(slice(0, heads))
    for at in range(0, heads, part):
        for a, b in zip(whole, run(slice(at, at + part))):
            assert torch.isfinite(b).all()
            assert torch.equal(a[:, at:at + part], b)


def test_many_keys_with_four_stages_in_segments_of_few_keys():
    """Segments of 1 to 300 keys beside a long one: every number of tiles that the ring can start with."""
    print("[gpu case] stages in segments", flush=True)
    heads, kv_heads, dim = 8, 8, 128
    lengths = [12000, 1, 64, 65, 128, 129, 192, 193, 256, 257, 300]
    assert launch_shape([1] * len(lengths), lengths, (heads, kv_heads), dim, causal=True) == (128, 4)
    gen = torch.Generator(device="cuda").manual_seed(12)
    total = sum(lengths)
    q, k, v = (torch.randn((n, h, dim), generator=gen, device="cuda").to(torch.bfloat16)
               for n, h in ((len(lengths), heads), (total, kv_heads), (total, kv_heads)))
    config = StreamingAttentionConfig(kv_chunk_tokens=192)
    plan = build_plan(q_heads=heads, kv_heads=kv_heads, head_dim=dim, dtype=torch.bfloat16, device="cuda",
                      max_q_tokens=len(lengths), max_kv_tokens=total, config=config)
    runner = StreamingAttentionRunner(plan, config)
    bounds = torch.tensor([0, *itertools.accumulate(lengths)])
    together, lse = runner(q, k, v, torch.arange(len(lengths) + 1), bounds, causal=True, return_lse=True)
    for s, n in enumerate(lengths):
        keys = slice(int(bounds[s]), int(bounds[s + 1]))
        alone, alone_lse = runner(q[s:s + 1], k[keys], v[keys], torch.tensor([0, 1]), torch.tensor([0, n]),
                                  causal=True, return_lse=True)
        assert torch.equal(together[s:s + 1], alone), n
        assert torch.equal(lse[:, s:s + 1], alone_lse), n
    torch.cuda.synchronize()
    runner.close()


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("q_heads,kv_heads,head_dim,dtype", [
    (32, 8, 128, torch.bfloat16),  # each XCD an eighth of the heads
    (12, 4, 128, torch.float16),   # workgroups dealt to the XCDs
    (32, 8, 64, torch.bfloat16),
    (40, 8, 96, torch.float16),
])
def test_packed_heads_with_four_stages_in_segments(q_heads, kv_heads, head_dim, dtype, causal):
    """Decoding steps and short continuations together (several query heads of
    a K/V head share a workgroup) equal each alone, which two stages run."""
    print(f"[gpu case] packed stages heads={q_heads}/{kv_heads} d={head_dim} {dtype} causal={causal}", flush=True)
    q_lengths = [1, 1, 3, 17, 1, 40, 2, 1]
    k_lengths = [n * 128 // head_dim * 8 // kv_heads for n in (1700, 64, 2301, 1500, 129, 1600, 1025, 2100)]
    assert launch_shape(q_lengths, k_lengths, (q_heads, kv_heads), head_dim, causal=causal) == (128, 4)
    cu_q, cu_k = ([0, *itertools.accumulate(x)] for x in (q_lengths, k_lengths))
    gen = torch.Generator(device="cuda").manual_seed(13)
    q, k, v = (torch.randn((n, h, head_dim), generator=gen, device="cuda").to(dtype)
               for n, h in ((cu_q[-1], q_heads), (cu_k[-1], kv_heads), (cu_k[-1], kv_heads)))
    config = StreamingAttentionConfig(kv_chunk_tokens=448)
    plan = build_plan(q_heads=q_heads, kv_heads=kv_heads, head_dim=head_dim, dtype=dtype, device="cuda",
                      max_q_tokens=cu_q[-1], max_kv_tokens=cu_k[-1], config=config)
    runner = StreamingAttentionRunner(plan, config)
    out, lse = runner(q, k, v, torch.tensor(cu_q), torch.tensor(cu_k), causal=causal, return_lse=True)
    for s, (n, keys) in enumerate(zip(q_lengths, k_lengths)):
        assert launch_shape([n], [keys], (q_heads, kv_heads), head_dim, causal=causal, causal_shift=keys - n)[1] == 2
        rows, cols = slice(cu_q[s], cu_q[s + 1]), slice(cu_k[s], cu_k[s + 1])
        alone, alone_lse = runner(q[rows], k[cols], v[cols], torch.tensor([0, n]), torch.tensor([0, keys]),
                                  causal=causal, return_lse=True)
        assert torch.equal(out[rows], alone), s
        assert torch.equal(lse[:, rows], alone_lse), s
    torch.cuda.synchronize()
    runner.close()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("rows,heads,causal,width", [
    (2048, 32, True, 128), (2048, 64, False, 256), (2100, 32, False, 384), (4100, 64, True, 384),
])
def test_transposed_v_at_every_width_equals_v_in_place(rows, heads, causal, width, dtype):
    print(f"[gpu case] transposed V rows={rows} heads={heads} causal={causal} {dtype}", flush=True)
    keys = 2111
    assert launch_shape([rows], [keys], (heads, heads // 32), 128, causal=causal, causal_shift=keys - rows,
                        kv_layout=TRANSPOSED_V)[0] == width
    gen = torch.Generator(device="cuda").manual_seed(14)
    q, k, v = (torch.randn((n, h, 128), generator=gen, device="cuda").to(dtype)
               for n, h in ((rows, heads), (keys, heads // 32), (keys, heads // 32)))
    results = []
    for limit in (None, 0):
        config = StreamingAttentionConfig(kv_chunk_tokens=512, resident_scratch_limit_bytes=limit)
        plan = build_plan(q_heads=heads, kv_heads=heads // 32, head_dim=128, dtype=dtype, device="cuda",
                          max_q_tokens=rows, max_kv_tokens=keys, config=config)
        runner = StreamingAttentionRunner(plan, config)
        stats = StreamingAttentionStats()
        results.append(runner(q, k, v, torch.tensor([0, rows]), torch.tensor([0, keys]), causal=causal,
                              return_lse=True, stats=stats))
        assert (stats.resident_scratch_bytes > 0) == (limit is None)
        torch.cuda.synchronize()
        runner.close()
    for a, b in zip(*results):
        assert torch.equal(a, b)
