"""GPU parity of the native gfx950 path against the CPU oracle.

Every case runs the product path (libseqattn_hip.so through the seqattn API
or its kernel boundary) and compares with oracle/seqattn_oracle.py on the same
seeded inputs.  Tolerances against the FP32-accumulated oracle:

* output max-abs <= 2e-2 and natural-log LSE max-abs <= 1e-3;
* output relative L2 error <= 5e-3 (the bound of the reference's paged GPU
  test, tests/test_paged_triton.py:87-88);
* every element within 2^-5 * (|ref| + rms(ref)).  Long sequences have tiny
  outputs (rms ~ sqrt(e / keys) for N(0,1) data), so the absolute bound alone
  would accept a wrong result of the right magnitude; a correct kernel's
  error is a few bf16 ulps of P and of the output (about 2^-9 relative).
"""

from __future__ import annotations

import numpy as np
import pytest
import torch

from oracle.seqattn_oracle import chunked_attention
from seqattn import StreamingAttentionConfig, StreamingAttentionRunner, StreamingAttentionStats, build_plan
from seqattn.kernels import finalize_attention, update_attention_state

pytestmark = pytest.mark.gpu

O_TOL = 2e-2
LSE_TOL = 1e-3
REL_L2_TOL = 5e-3
SCALED_TOL = 2.0**-5


def announce(name: str) -> None:
    print(f"[gpu case] {name}", flush=True)


def pinned_randn(shape, dtype, gen, scale=1.0):
    return (torch.randn(shape, generator=gen) * scale).to(dtype).pin_memory()


def oracle(q, k, v, cu_q, cu_k, *, q_chunk, kv_chunk, causal, scale=None, rows=None):
    return chunked_attention(
        q.float().numpy(), k.float().numpy(), v.float().numpy(),
        np.asarray(cu_q), np.asarray(cu_k),
        q_chunk_tokens=q_chunk, kv_chunk_tokens=kv_chunk, softmax_scale=scale, causal=causal, rows=rows,
    )


def check(out, lse, ref_o, ref_l, rows=None):
    o = out.float().numpy()
    l = lse.float().cpu().numpy()
    if rows is not None:
        o, ref_o = o[rows], ref_o[rows]
        l, ref_l = l[:, rows], ref_l[:, rows]
    assert np.isfinite(o).all()
    diff = np.abs(o - ref_o)
    err_o = float(diff.max())
    ref_norm = float(np.sqrt(np.square(ref_o, dtype=np.float64).sum()))
    rel_l2 = float(np.sqrt(np.square(diff, dtype=np.float64).sum())) / ref_norm if ref_norm > 0 else 0.0
    rms = ref_norm / np.sqrt(ref_o.size) if ref_o.size else 0.0
    scaled = float((diff / (np.abs(ref_o) + rms)).max()) if rms > 0 else 0.0
    finite = np.isfinite(ref_l)
    assert np.array_equal(np.isfinite(l), finite), "LSE -inf pattern differs"
    err_l = float(np.abs(l[finite] - ref_l[finite]).max()) if finite.any() else 0.0
    print(f"    max|dO|={err_o:.3e} relL2={rel_l2:.3e} scaled={scaled:.3e} max|dLSE|={err_l:.3e}", flush=True)
    assert err_o <= O_TOL, err_o
    assert rel_l2 <= REL_L2_TOL, rel_l2
    assert scaled <= SCALED_TOL, scaled
    assert err_l <= LSE_TOL, err_l


def run(q, k, v, cu_q, cu_k, config, *, causal=False, scale=None):
    plan = build_plan(q_heads=q.shape[1], kv_heads=k.shape[1], head_dim=q.shape[2], dtype=q.dtype,
                      device="cuda", max_q_tokens=q.shape[0], max_kv_tokens=k.shape[0], config=config)
    runner = StreamingAttentionRunner(plan, config)
    out, lse = runner(q, k, v, cu_q, cu_k, causal=causal, softmax_scale=scale, return_lse=True)
    return out, lse, runner


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("q_heads,kv_heads", [(4, 4), (8, 2)])
def test_matches_oracle_at_reference_test_shapes(dtype, causal, q_heads, kv_heads):
    # The shapes of the reference's tests/test_triton.py:17-57 (empty middle segment,
    # chunk sizes that divide nothing).
    announce(f"reference shapes {dtype} causal={causal} heads={q_heads}/{kv_heads}")
    gen = torch.Generator().manual_seed(17)
    q = pinned_randn((73, q_heads, 64), dtype, gen)
    k = pinned_randn((89, kv_heads, 64), dtype, gen)
    v = pinned_randn((89, kv_heads, 64), dtype, gen)
    cu_q = torch.tensor([0, 31, 31, 73], dtype=torch.int32)
    cu_k = torch.tensor([0, 37, 37, 89], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="triton", q_chunk_tokens=23, kv_chunk_tokens=19,
                                      block_m=32, block_n=32)
    out, lse, _ = run(q, k, v, cu_q, cu_k, config, causal=causal)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=23, kv_chunk=19, causal=causal)
    check(out, lse, ref_o, ref_l)


# Every padded head_dim (32, 64, 128, 256) and its edges, including head_dims
# that end inside a 16-wide d block (40, 72, 104, 120) or a 32-wide d step (80).
@pytest.mark.parametrize("head_dim", [16, 32, 40, 48, 64, 72, 80, 96, 104, 120, 128, 136, 200, 256])
@pytest.mark.parametrize("causal", [False, True])
def test_head_dims_ragged_chunks(head_dim, causal):
    announce(f"head_dim={head_dim} causal={causal}")
    gen = torch.Generator().manual_seed(100 + head_dim)
    q = pinned_randn((333, 6, head_dim), torch.bfloat16, gen)
    k = pinned_randn((290, 3, head_dim), torch.bfloat16, gen)
    v = pinned_randn((290, 3, head_dim), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 1, 200, 333], dtype=torch.int32)
    cu_k = torch.tensor([0, 70, 210, 290], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=130, kv_chunk_tokens=70, num_kv_buffers=3)
    out, lse, _ = run(q, k, v, cu_q, cu_k, config, causal=causal, scale=0.11)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=128, kv_chunk=64, causal=causal, scale=0.11)
    check(out, lse, ref_o, ref_l)


def test_device_consumer_q_reuse_matches_separate_output_path():
    # Mirrors the reference's tests/test_triton.py:94-145: bit-identical outputs.
    announce("device consumer Q reuse")
    gen = torch.Generator().manual_seed(29)
    q = pinned_randn((83, 4, 32), torch.bfloat16, gen)
    k = pinned_randn((91, 2, 32), torch.bfloat16, gen)
    v = pinned_randn((91, 2, 32), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 37, 83], dtype=torch.int32)
    cu_k = torch.tensor([0, 41, 91], dtype=torch.int32)

    def identity_consumer(attention, start, stop):
        del start, stop
        return attention.reshape(-1, 4, 32)

    outputs, runners = [], []
    for output_mode in ("host", "device_consumer"):
        config = StreamingAttentionConfig(backend="triton", q_chunk_tokens=31, kv_chunk_tokens=32,
                                          block_m=16, block_n=16, num_output_buffers=2, output_mode=output_mode)
        plan = build_plan(q_heads=4, kv_heads=2, head_dim=32, dtype=q.dtype, device="cuda",
                          max_q_tokens=q.shape[0], max_kv_tokens=k.shape[0], config=config)
        runner = StreamingAttentionRunner(plan, config)
        out = torch.empty_like(q).pin_memory()
        runner.run_with_device_output(q, k, v, cu_q, cu_k, output_transform=identity_consumer, out=out, causal=True)
        outputs.append(out)
        runners.append(runner)
    torch.testing.assert_close(outputs[1], outputs[0], atol=0, rtol=0)
    assert len(runners[0]._workspace.output) == 2
    assert runners[1]._workspace.output == []
    ref_o, _ = oracle(q, k, v, cu_q, cu_k, q_chunk=31, kv_chunk=32, causal=True)
    assert float(np.abs(outputs[0].float().numpy() - ref_o).max()) <= O_TOL


def test_host_aliased_and_device_resident_outputs_are_bit_identical_to_host_mode():
    announce("host_aliased / device out")
    gen = torch.Generator().manual_seed(31)
    q = pinned_randn((700, 8, 128), torch.bfloat16, gen)
    k = pinned_randn((650, 8, 128), torch.bfloat16, gen)
    v = pinned_randn((650, 8, 128), torch.bfloat16, gen)
    cu = torch.tensor([0, 300, 700], dtype=torch.int32)
    cu_k = torch.tensor([0, 250, 650], dtype=torch.int32)
    results = []
    for mode in ("host", "host_aliased"):
        config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=256, kv_chunk_tokens=128, output_mode=mode)
        out, lse, runner = run(q, k, v, cu, cu_k, config)
        results.append((out, lse))
    device_out = torch.empty(q.shape, dtype=q.dtype, device="cuda")
    runner(q, k, v, cu, cu_k, out=device_out)
    torch.testing.assert_close(results[1][0], results[0][0], atol=0, rtol=0)
    torch.testing.assert_close(results[1][1], results[0][1], atol=0, rtol=0)
    torch.testing.assert_close(device_out.cpu(), results[0][0], atol=0, rtol=0)
    ref_o, ref_l = oracle(q, k, v, cu, cu_k, q_chunk=256, kv_chunk=128, causal=False)
    check(results[0][0], results[0][1], ref_o, ref_l)


@pytest.mark.parametrize("causal", [False, True])
def test_host_aliased_piecewise_boundaries_are_bit_identical_to_host_mode(causal):
    """host_aliased runs work each pass boundary in row pieces of the block
    (the last chunk per piece, the output copied out and the next block's Q
    rows copied in piece by piece, the first chunk per piece).  Blocks of 3-4
    workgroup tiles give 3-4 pieces; the third segment has fewer keys than
    one chunk, so its passes are a single (initializing, output-writing)
    chunk; the second has fewer keys than queries, so under the causal rule
    its first 100 rows see no key.  GQA 8/2, bf16."""
    announce(f"host_aliased piecewise boundaries causal={causal}")
    gen = torch.Generator().manual_seed(43)
    cu_q = torch.tensor([0, 2000, 3300, 3800], dtype=torch.int32)
    cu_k = torch.tensor([0, 1800, 3000, 3200], dtype=torch.int32)
    q = pinned_randn((3800, 8, 128), torch.bfloat16, gen)
    k = pinned_randn((3200, 2, 128), torch.bfloat16, gen)
    v = pinned_randn((3200, 2, 128), torch.bfloat16, gen)
    results = []
    for mode in ("host", "host_aliased"):
        config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=1536, kv_chunk_tokens=256, output_mode=mode)
        stats = StreamingAttentionStats()
        plan = build_plan(q_heads=8, kv_heads=2, head_dim=128, dtype=torch.bfloat16, device="cuda",
                          max_q_tokens=3800, max_kv_tokens=3200, config=config)
        runner = StreamingAttentionRunner(plan, config)
        out, lse = runner(q, k, v, cu_q, cu_k, causal=causal, return_lse=True, stats=stats)
        results.append((out, lse, stats))
        runner.close()
    (out_h, lse_h, st_h), (out_a, lse_a, st_a) = results
    torch.testing.assert_close(out_a, out_h, atol=0, rtol=0)
    torch.testing.assert_close(lse_a, lse_h, atol=0, rtol=0)
    assert st_a.h2d_bytes == st_h.h2d_bytes and st_a.d2h_bytes == st_h.d2h_bytes == 3800 * 8 * 128 * 2
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=1536, kv_chunk=256, causal=causal)
    check(out_a, lse_a, ref_o, ref_l)


@pytest.mark.parametrize("kv_chunk", [96, 128])
@pytest.mark.parametrize("causal", [False, True])
def test_device_resident_inputs_are_bit_identical_to_streamed(causal, kv_chunk):
    """HBM-resident Q/K/V give the pinned-host streamed run's output and LSE
    bit for bit.  With a 128-key chunk (a multiple of the 64-key tile) each Q
    block is one launch over all keys that merges the row sums at every chunk
    boundary; with 96 it is one launch per chunk, as in the streamed run."""
    announce(f"device-resident inputs causal={causal} kv_chunk={kv_chunk}")
    gen = torch.Generator().manual_seed(37)
    q = pinned_randn((611, 8, 128), torch.bfloat16, gen)
    k = pinned_randn((540, 2, 128), torch.bfloat16, gen)
    v = pinned_randn((540, 2, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 200, 200, 611], dtype=torch.int32)
    cu_k = torch.tensor([0, 150, 150, 540], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=160, kv_chunk_tokens=kv_chunk)
    out, lse, runner = run(q, k, v, cu_q, cu_k, config, causal=causal)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out_d, lse_d = runner(qd, kd, vd, cu_q, cu_k, causal=causal, return_lse=True)
    torch.cuda.synchronize()
    assert out_d.device.type == "cuda"
    torch.testing.assert_close(out_d.cpu(), out, atol=0, rtol=0)
    torch.testing.assert_close(lse_d.cpu(), lse, atol=0, rtol=0)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=160, kv_chunk=kv_chunk, causal=causal)
    check(out_d.cpu(), lse_d, ref_o, ref_l)


@pytest.mark.parametrize("dtype,head_dim,q_heads,kv_heads", [
    (torch.float16, 128, 4, 4),
    (torch.bfloat16, 64, 6, 2),
    (torch.bfloat16, 96, 4, 1),
    (torch.bfloat16, 256, 2, 1),
    (torch.bfloat16, 128, 12, 4),  # causal blocks dealt to XCDs in a launch of more than 8 heads
])
def test_fused_resident_launch_matches_streamed_at_every_geometry(dtype, head_dim, q_heads, kv_heads):
    """With device inputs and a K/V chunk that is a multiple of 64, the
    segments are one launch that finalizes its rows in the epilogue, V read in
    place.  At every padded head_dim and both 16-bit dtypes it gives the
    pinned-host streamed run's output and LSE bit for bit, causal, including
    the first segment's 200 queries that see no key (output 0, LSE -inf)."""
    announce(f"fused resident launch {dtype} d={head_dim} heads={q_heads}/{kv_heads}")
    gen = torch.Generator().manual_seed(41)
    q = pinned_randn((700, q_heads, head_dim), dtype, gen)
    k = pinned_randn((900, kv_heads, head_dim), dtype, gen)
    v = pinned_randn((900, kv_heads, head_dim), dtype, gen)
    cu_q = torch.tensor([0, 300, 700], dtype=torch.int32)
    cu_k = torch.tensor([0, 100, 900], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=192, kv_chunk_tokens=128)
    out, lse, runner = run(q, k, v, cu_q, cu_k, config, causal=True)
    out_d, lse_d = runner(q.cuda(), k.cuda(), v.cuda(), cu_q, cu_k, causal=True, return_lse=True)
    torch.cuda.synchronize()
    torch.testing.assert_close(out_d.cpu(), out, atol=0, rtol=0)
    torch.testing.assert_close(lse_d.cpu(), lse, atol=0, rtol=0)
    assert torch.isneginf(lse_d[:, :200]).all() and (out_d[:200] == 0).all()
    assert runner._workspace.resident_scratch is None  # too few queries for a transposed copy of V
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=192, kv_chunk=128, causal=True)
    check(out_d.cpu(), lse_d, ref_o, ref_l)


@pytest.mark.parametrize("causal", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_transposed_v_of_large_segments_matches_streamed(causal, dtype):
    """From 65,536 queries x query heads per K/V head a head_dim-128 segment
    reads V through a transposed copy, one scratch for consecutive segments:
    the first, third and fourth here (odd numbers of keys, the fourth with
    fewer than queries), in between one that reads it in place."""
    announce(f"transposed V large segments causal={causal} {dtype}")
    gen = torch.Generator().manual_seed(71)
    cu_q = torch.tensor([0, 2048, 2148, 4248, 6348], dtype=torch.int32)
    cu_k = torch.tensor([0, 2111, 2400, 5201, 6500], dtype=torch.int32)
    q = pinned_randn((6348, 64, 128), dtype, gen)
    k = pinned_randn((6500, 2, 128), dtype, gen)
    v = pinned_randn((6500, 2, 128), dtype, gen)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=2048, kv_chunk_tokens=1024)
    out, lse, runner = run(q, k, v, cu_q, cu_k, config, causal=causal)
    stats = StreamingAttentionStats()
    out_d, lse_d = runner(q.cuda(), k.cuda(), v.cuda(), cu_q, cu_k, causal=causal, return_lse=True, stats=stats)
    torch.cuda.synchronize()
    assert stats.resident_scratch_bytes == 2 * 128 * 2816 * 2  # the third segment's 2,801 keys
    assert torch.equal(out_d.cpu(), out)
    assert torch.equal(lse_d.cpu(), lse.cpu())


def test_runs_that_read_v_in_place_allocate_no_scratch():
    """Decoding steps and continuations of a long context hold no transposed
    copy of V; the run of many queries between them does."""
    announce("resident scratch")
    gen = torch.Generator(device="cuda").manual_seed(73)
    q, k, v = (torch.randn((n, h, 128), generator=gen, device="cuda").to(torch.bfloat16)
               for n, h in ((2100, 32), (5000, 1), (5000, 1)))
    config = StreamingAttentionConfig(backend="hip", kv_chunk_tokens=1024)
    plan = build_plan(q_heads=32, kv_heads=1, head_dim=128, dtype=torch.bfloat16, device="cuda", max_q_tokens=2100,
                      max_kv_tokens=5000, config=config)
    runner = StreamingAttentionRunner(plan, config)
    keys = torch.tensor([0, 5000])
    for rows, scratch in ((1, 0), (1009, 0), (2048, 128 * 5056 * 2), (7, 0)):
        stats = StreamingAttentionStats()
        runner(q[:rows], k, v, torch.tensor([0, rows]), keys, causal=True, stats=stats)
        assert stats.resident_scratch_bytes == scratch
        if rows <= 1009 and rows != 7:
            assert runner._workspace.resident_scratch is None
    torch.cuda.synchronize()
    runner.close()


@pytest.mark.parametrize("causal", [False, True])
def test_transposed_v_pads_short_segments_exactly(causal):
    """The copy of V is padded with zero keys to whole 64-key tiles.  Segments
    of 3 keys, none, exactly one tile and two tiles and a key, each with
    enough queries to take the copy, give the streamed run's output and LSE bit
    for bit."""
    announce(f"transposed V short segments causal={causal}")
    gen = torch.Generator().manual_seed(47)
    cu_q = torch.tensor([0, 2048, 2048, 4097, 6197], dtype=torch.int32)
    cu_k = torch.tensor([0, 3, 3, 67, 196], dtype=torch.int32)
    q = pinned_randn((6197, 32, 128), torch.bfloat16, gen)
    k = pinned_randn((196, 1, 128), torch.bfloat16, gen)
    v = pinned_randn((196, 1, 128), torch.bfloat16, gen)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=1024, kv_chunk_tokens=64)
    out, lse, runner = run(q, k, v, cu_q, cu_k, config, causal=causal)
    stats = StreamingAttentionStats()
    out_d, lse_d = runner(q.cuda(), k.cuda(), v.cuda(), cu_q, cu_k, causal=causal, return_lse=True, stats=stats)
    torch.cuda.synchronize()
    assert stats.resident_scratch_bytes == 128 * 192 * 2
    torch.testing.assert_close(out_d.cpu(), out, atol=0, rtol=0)
    torch.testing.assert_close(lse_d.cpu(), lse, atol=0, rtol=0)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=1024, kv_chunk=64, causal=causal)
    # Under the causal rule most queries see no key (their zeros and -inf were
    # compared above): the file's bounds scale with the rms of the rows that do.
    seen = np.flatnonzero(np.isfinite(ref_l[0]))
    check(out_d.cpu(), lse_d, ref_o, ref_l, rows=seen)


@pytest.mark.parametrize("num_kv", [1, 3])
@pytest.mark.parametrize("causal", [False, True])
def test_split_chunk_updates_on_two_streams_are_bit_identical(causal, num_kv):
    """Streamed Q blocks of two workgroup tiles or more (768 rows at head_dim
    128) apply each K/V chunk with two launches, one per half of the rows, on
    two streams.  With a one-slot ring
    the next copy must wait for both halves; with three slots the halves run
    ahead of each other.  Host output, device-consumer output and the
    HBM-resident single launch agree bit for bit."""
    announce(f"split chunk updates causal={causal} num_kv={num_kv}")
    gen = torch.Generator().manual_seed(43)
    q = pinned_randn((1400, 4, 128), torch.bfloat16, gen)
    k = pinned_randn((1300, 2, 128), torch.bfloat16, gen)
    v = pinned_randn((1300, 2, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 1100, 1400], dtype=torch.int32)
    cu_k = torch.tensor([0, 1000, 1300], dtype=torch.int32)
    results, runners = [], []
    for output_mode in ("host", "device_consumer"):
        config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=1024, kv_chunk_tokens=256,
                                          num_kv_buffers=num_kv, output_mode=output_mode)
        plan = build_plan(q_heads=4, kv_heads=2, head_dim=128, dtype=q.dtype, device="cuda",
                          max_q_tokens=q.shape[0], max_kv_tokens=k.shape[0], config=config)
        runner = StreamingAttentionRunner(plan, config)
        out = torch.empty_like(q).pin_memory()
        if output_mode == "host":
            runner(q, k, v, cu_q, cu_k, out=out, causal=causal)
        else:
            runner.run_with_device_output(q, k, v, cu_q, cu_k, output_transform=lambda a, s, e: a.reshape(-1, 4, 128),
                                          out=out, causal=causal)
        torch.cuda.synchronize()
        results.append(out)
        runners.append(runner)
    out_d = runners[0](q.cuda(), k.cuda(), v.cuda(), cu_q, cu_k, causal=causal)
    torch.cuda.synchronize()
    torch.testing.assert_close(results[1], results[0], atol=0, rtol=0)
    torch.testing.assert_close(out_d.cpu(), results[0], atol=0, rtol=0)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=1024, kv_chunk=256, causal=causal)
    check(results[0], torch.from_numpy(ref_l), ref_o, ref_l)


def test_runners_share_one_copy_stream_pair_and_still_agree():
    """Every workspace on a device uses the same H2D / D2H streams (fresh
    streams per runner can land on the compute stream's hardware queue).
    Runners interleaved on the shared pair give the results of a lone one."""
    announce("shared copy streams")
    gen = torch.Generator().manual_seed(67)
    q = pinned_randn((400, 4, 128), torch.bfloat16, gen)
    k = pinned_randn((380, 4, 128), torch.bfloat16, gen)
    v = pinned_randn((380, 4, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 400], dtype=torch.int32)
    cu_k = torch.tensor([0, 380], dtype=torch.int32)
    configs = [StreamingAttentionConfig(backend="hip", q_chunk_tokens=qc, kv_chunk_tokens=kc)
               for qc, kc in ((64, 48), (128, 96), (96, 64))]
    runners, outs = [], []
    for config in configs:
        out, lse, runner = run(q, k, v, cu_q, cu_k, config)
        runners.append(runner)
        outs.append((out, lse))
    streams = {(r._workspace.h2d_stream.cuda_stream, r._workspace.d2h_stream.cuda_stream) for r in runners}
    assert len(streams) == 1, streams
    h2d, d2h = next(iter(streams))
    assert h2d != d2h
    # Second round, runners alternating on the shared pair.
    for runner, (out, lse) in zip(runners, outs):
        out2, lse2 = runner(q, k, v, cu_q, cu_k, return_lse=True)
        torch.testing.assert_close(out2, out, atol=0, rtol=0)
        torch.testing.assert_close(lse2, lse, atol=0, rtol=0)
    for (out, lse), config in zip(outs, configs):
        ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=config.q_chunk_tokens,
                              kv_chunk=config.kv_chunk_tokens, causal=False)
        check(out, lse, ref_o, ref_l)


@pytest.mark.parametrize("causal", [False, True])
def test_one_and_two_output_slots_give_identical_results(causal):
    """With one output slot the pipeline alternates the Q block buffer and the
    slot between passes and copies the next Q block in pieces between K/V
    chunks; with two slots it keeps the executor's order.  Many passes over
    three segments (one empty) must agree bit for bit and match the oracle."""
    announce(f"output slots 1 vs 2 causal={causal}")
    gen = torch.Generator().manual_seed(61)
    q = pinned_randn((701, 4, 128), torch.bfloat16, gen)
    k = pinned_randn((650, 2, 128), torch.bfloat16, gen)
    v = pinned_randn((650, 2, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 290, 290, 701], dtype=torch.int32)
    cu_k = torch.tensor([0, 260, 260, 650], dtype=torch.int32)
    results = []
    for slots in (1, 2):
        config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=64, kv_chunk_tokens=48,
                                          num_output_buffers=slots)
        out, lse, runner = run(q, k, v, cu_q, cu_k, config, causal=causal)
        assert runner.plan.num_output_buffers == slots
        # A second call on the same runner reuses the buffers in their new roles.
        out2, lse2 = runner(q, k, v, cu_q, cu_k, causal=causal, return_lse=True)
        torch.testing.assert_close(out2, out, atol=0, rtol=0)
        torch.testing.assert_close(lse2, lse, atol=0, rtol=0)
        results.append((out, lse))
    torch.testing.assert_close(results[0][0], results[1][0], atol=0, rtol=0)
    torch.testing.assert_close(results[0][1], results[1][1], atol=0, rtol=0)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=64, kv_chunk=48, causal=causal)
    check(results[0][0], results[0][1], ref_o, ref_l)


@pytest.mark.parametrize("scale", [-0.2, 0.0, 1e-3])
def test_negative_zero_and_tiny_softmax_scales(scale):
    """The kernel folds a negative scale into the sign of Q and treats a zero
    scale as 1e-30; both must reproduce softmax(scale * QK^T) V."""
    announce(f"softmax scale {scale}")
    gen = torch.Generator().manual_seed(53)
    q = pinned_randn((300, 4, 128), torch.bfloat16, gen)
    k = pinned_randn((500, 2, 128), torch.bfloat16, gen)
    v = pinned_randn((500, 2, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 100, 300], dtype=torch.int32)
    cu_k = torch.tensor([0, 240, 500], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=128, kv_chunk_tokens=160)
    out, lse, _ = run(q, k, v, cu_q, cu_k, config, causal=True, scale=scale)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=128, kv_chunk=160, causal=True, scale=scale)
    check(out, lse, ref_o, ref_l)


def test_repeated_runs_are_bit_identical():
    """Many workgroups per head and many K/V tiles per launch: three runs of
    the same inputs must agree bit for bit (a race between the LDS DMA of one
    wave and the reads of another shows up as run-to-run differences)."""
    announce("determinism")
    gen = torch.Generator().manual_seed(43)
    q = pinned_randn((4096, 16, 128), torch.bfloat16, gen)
    k = pinned_randn((6000, 16, 128), torch.bfloat16, gen)
    v = pinned_randn((6000, 16, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 4096], dtype=torch.int32)
    cu_k = torch.tensor([0, 6000], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=4096, kv_chunk_tokens=3000)
    out, lse, runner = run(q, k, v, cu_q, cu_k, config)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    for _ in range(2):
        again, lse_again = runner(qd, kd, vd, cu_q, cu_k, return_lse=True)
        torch.cuda.synchronize()
        torch.testing.assert_close(again.cpu(), out, atol=0, rtol=0)
        torch.testing.assert_close(lse_again.cpu(), lse, atol=0, rtol=0)
    rows = np.arange(0, 4096, 37)
    ref_o, ref_l = oracle(q, k, v, cu_q, cu_k, q_chunk=4096, kv_chunk=3000, causal=False, rows=rows)
    check(out, lse, ref_o, ref_l, rows=rows)


def test_results_do_not_depend_on_the_q_block_decomposition():
    """Each query's online-softmax trajectory depends only on its own logits,
    so different resident Q blocks give bit-identical rows."""
    announce("q block independence")
    gen = torch.Generator().manual_seed(47)
    q = pinned_randn((900, 4, 128), torch.bfloat16, gen, scale=2.0)
    k = pinned_randn((1000, 4, 128), torch.bfloat16, gen, scale=2.0)
    v = pinned_randn((1000, 4, 128), torch.bfloat16, gen)
    cu_q = torch.tensor([0, 900], dtype=torch.int32)
    cu_k = torch.tensor([0, 1000], dtype=torch.int32)
    outputs = []
    for q_chunk in (900, 257, 96):
        config = StreamingAttentionConfig(backend="hip", q_chunk_tokens=q_chunk, kv_chunk_tokens=320)
        out, lse, _ = run(q, k, v, cu_q, cu_k, config, causal=True)
        outputs.append((out, lse))
    for out, lse in outputs[1:]:
        torch.testing.assert_close(out, outputs[0][0], atol=0, rtol=0)
        torch.testing.assert_close(lse, outputs[0][1], atol=0, rtol=0)


def test_runner_reuse_has_bounded_allocator_growth():
    announce("allocator growth")
    gen = torch.Generator().manual_seed(19)
    q = pinned_randn((257, 4, 64), torch.bfloat16, gen)
    k = pinned_randn((257, 4, 64), torch.bfloat16, gen)
    v = pinned_randn((257, 4, 64), torch.bfloat16, gen)
    cu = torch.tensor([0, 257], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="triton", q_chunk_tokens=128, kv_chunk_tokens=96, block_m=32, block_n=32)
    plan = build_plan(q_heads=4, kv_heads=4, head_dim=64, dtype=q.dtype, device="cuda",
                      max_q_tokens=257, max_kv_tokens=257, config=config)
    runner = StreamingAttentionRunner(plan, config)
    first = runner(q, k, v, cu, cu)
    torch.cuda.synchronize()
    baseline = torch.cuda.memory_allocated()
    for _ in range(20):
        again = runner(q, k, v, cu, cu)
    torch.cuda.synchronize()
    assert torch.cuda.memory_allocated() <= baseline + 2 * 2**20
    torch.testing.assert_close(again, first, atol=0, rtol=0)


def test_kernel_boundary_on_device_tensors_with_outliers():
    """Resident mode through the kernel API: Q/K/V already in HBM, one Q block,
    K/V applied in uneven chunks; 1% of key rows scaled x8 (softmax-merge stress)."""
    announce("kernel API outliers")
    gen = torch.Generator().manual_seed(41)
    n_q, n_k, heads, d = 1000, 1500, 4, 128
    q = torch.randn((n_q, heads, d), generator=gen).to(torch.bfloat16)
    k = torch.randn((n_k, heads, d), generator=gen)
    idx = torch.randperm(n_k, generator=gen)[: n_k // 100]
    k[idx] *= 8
    k = k.to(torch.bfloat16)
    v = torch.randn((n_k, heads, d), generator=gen).to(torch.bfloat16)
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    m = torch.empty((n_q, heads), device="cuda")
    l = torch.empty_like(m)
    acc = torch.empty((n_q, heads, d), device="cuda")
    scale = d**-0.5
    starts = [0, 700, 701, 1200]
    stops = starts[1:] + [n_k]
    for i, (s, e) in enumerate(zip(starts, stops)):
        update_attention_state(qd, kd[s:e], vd[s:e], m, l, acc, q_tokens=n_q, kv_tokens=e - s,
                               q_local_offset=0, kv_local_offset=s, causal_shift=n_k - n_q,
                               softmax_scale=scale, causal=False, initialize=i == 0)
    out = torch.empty((n_q, heads, d), dtype=torch.bfloat16, device="cuda")
    lse = torch.empty((heads, n_q), device="cuda")
    finalize_attention(acc, l, out, q_tokens=n_q, running_max=m, lse=lse)
    torch.cuda.synchronize()
    ref_o, ref_l = oracle(q, k, v, [0, n_q], [0, n_k], q_chunk=n_q, kv_chunk=n_k, causal=False)
    check(out.cpu(), lse, ref_o, ref_l)


def test_65k_tokens_32_heads_streamed_1gib_and_resident():
    """65,536 tokens x 32 heads x 128, bf16, N(0,1) seeded per 4,096-token
    chunk as the reference benchmark: streamed with a 1 GiB workspace and
    4,096-token K/V chunks (sampled rows vs the oracle), then fully resident
    in HBM (bit-identical to the streamed run)."""
    announce("65k x 32h streamed 1GiB")
    from oracle.seqattn_oracle import seeded_normal_chunks

    n, heads, d = 65536, 32, 128
    q, k, v = (seeded_normal_chunks(n, heads, d, seed=0, tensor_index=i).pin_memory() for i in range(3))
    cu = torch.tensor([0, n], dtype=torch.int32)
    config = StreamingAttentionConfig(backend="hip", workspace_budget_bytes=2**30, kv_chunk_tokens=4096)
    out, lse, runner = run(q, k, v, cu, cu, config)
    rng = np.random.default_rng(0)
    rows = np.unique(np.concatenate([[0, n // 4, n // 2, 3 * n // 4, n - 1], rng.choice(n, 251, replace=False)]))
    ref_o, ref_l = oracle(q, k, v, [0, n], [0, n], q_chunk=runner.plan.q_chunk_tokens, kv_chunk=4096,
                          causal=False, rows=rows)
    check(out, lse, ref_o, ref_l, rows=rows)

    announce("65k x 32h fully resident in HBM")
    qd, kd, vd = q.cuda(), k.cuda(), v.cuda()
    out_d, lse_d = runner(qd, kd, vd, cu, cu, return_lse=True)
    torch.cuda.synchronize()
    torch.testing.assert_close(out_d.cpu(), out, atol=0, rtol=0)
    torch.testing.assert_close(lse_d.cpu(), lse, atol=0, rtol=0)
