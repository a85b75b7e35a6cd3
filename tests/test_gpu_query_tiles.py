"""The update kernel's workgroup widths (128, 256 and 384 queries) give the same bits.

A launch picks its width for speed; a query's online softmax must not depend
on which other queries share its workgroup.  Each launch below is wide enough
to take a wide workgroup (64 heads; the last block is partly filled) and is
repeated in slices of at most 100 queries, which take the narrow one.
"""

from __future__ import annotations

import itertools

import pytest
import torch

from seqattn import StreamingAttentionConfig, StreamingAttentionRunner, build_plan
from seqattn.kernels import update_attention_state, update_attention_state_int8

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("head_dim,rows,int8", [
    (32, 1000, False), (64, 1000, False), (64, 1000, True), (96, 1000, False), (128, 1000, False),
    (128, 1500, False), (128, 1500, True), (256, 1000, False),
])
def test_workgroup_widths_give_the_same_state(head_dim, rows, int8, causal):
    print(f"[gpu case] widths d={head_dim} rows={rows} int8={int8} causal={causal}", flush=True)
    gen = torch.Generator(device="cuda").manual_seed(5)
    heads, kv_heads, keys = 64, 8, 1530
    q = torch.randn((rows, heads, head_dim), generator=gen, device="cuda").to(torch.bfloat16)
    if int8:
        k, v = (torch.randint(-127, 128, (keys, kv_heads, head_dim), generator=gen, device="cuda", dtype=torch.int8)
                for _ in range(2))
        scales = [torch.rand((-(-keys // 64), kv_heads), generator=gen, device="cuda").mul_(0.05).half()
                  for _ in range(2)]
    else:
        k, v = (torch.randn((keys, kv_heads, head_dim), generator=gen, device="cuda").to(torch.bfloat16)
                for _ in range(2))

    def run(start, stop, m, l, acc):
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
    """300 heads are more workgroups than CUs (two LDS stages); 150 of them are fewer (four: over 32 MB of K and V)."""
    print(f"[gpu case] stages d={head_dim} causal={causal} tail={tail}", flush=True)
    heads, part, rows = 300, 150, 3
    keys = -(-(33 << 20) // (4 * part * head_dim)) // 64 * 64 + 64 + tail
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
    lengths = [8300, 1, 64, 65, 128, 129, 192, 193, 256, 257, 300]
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
