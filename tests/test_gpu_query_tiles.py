"""The update kernel's workgroup widths (128, 256 and 384 queries) give the same bits.

A launch picks its width for speed; a query's online softmax must not depend
on which other queries share its workgroup.  Each launch below is wide enough
to take a wide workgroup (64 heads; the last block is partly filled) and is
repeated in slices of at most 100 queries, which take the narrow one.
"""

from __future__ import annotations

import pytest
import torch

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
