"""The calls this framework is used for, as measurable cases.

Every case goes through a public entry point of ``seqattn``, as a program
would call it.  The kinds:

* ``resident``: a kept ``StreamingAttentionRunner`` on Q/K/V in HBM (one or
  many packed segments, LSE returned): a serving or embedding program's
  prefill, the continuation of a long context (few queries, many keys) and
  decoding (one query per sequence).
* ``host``: page-locked host Q/K/V in, page-locked host output, through the
  functional API (``streaming_attn_func``) or a kept runner with a workspace
  budget and a schedule: the framework's main use, sequences whose Q/K/V do
  not stay in HBM.
* ``chunks``: the kernel API (``update_attention_state`` or its INT8 K/V
  variant, then ``finalize_attention``), K/V arriving in chunks: a program
  that runs its own schedule.
* ``paged``: ``PagedAttentionRunner`` over page-locked pages, output in HBM.

Inputs are N(0, 1), the distribution of the repository's tests and benchmark;
``outliers`` scales 1% of the key rows by 8, as its paged workload does.
"""

from __future__ import annotations

import itertools
import random
import sys
from pathlib import Path

import torch

ROOT = Path(__file__).resolve().parents[1]
if str(ROOT / "stream-attn_amd") not in sys.path:
    sys.path.insert(0, str(ROOT / "stream-attn_amd"))

import seqattn  # noqa: E402
from seqattn.kernels import finalize_attention, update_attention_state, update_attention_state_int8  # noqa: E402

DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16}
QUANT_GROUP = 64  # tokens per INT8 scale


def _case(kind, segments, q_tokens, kv_tokens, q_heads, kv_heads, head_dim, *, name=None, dtype="bf16", causal=False,
          ragged=False, outliers=False, entry="runner", schedule="q_blocks", budget_mib=0, kv_chunk=0, page=0,
          int8=False):
    case = dict(kind=kind, segments=segments, q_tokens=q_tokens, kv_tokens=kv_tokens, q_heads=q_heads,
                kv_heads=kv_heads, head_dim=head_dim, dtype=dtype, causal=causal, ragged=ragged, outliers=outliers,
                entry=entry, schedule=schedule, budget_mib=budget_mib, kv_chunk=kv_chunk, page=page, int8=int8)
    if name is not None:
        case["name"] = name
    return case


def listed():
    return [
        # One short sequence, 8 heads of 64: the smallest call, latency.
        _case("resident", 1, 512, 512, 8, 8, 64, name="resident_512x8_d64"),
        # A dense batch of equal sequences through a kept runner (an encoder's
        # layer).
        _case("resident", 6, 6 * 2048, 6 * 2048, 16, 16, 64, name="resident_batch6_2048x16_d64"),
        # A packed prefill batch of ragged sequences, grouped-query heads.
        _case("resident", 11, 20011, 20011, 32, 8, 128, name="resident_ragged11_causal_gqa_fp16", dtype="fp16",
              causal=True, ragged=True),
        # The next 1,009 tokens of a sequence with 61,312 keys in HBM.
        _case("resident", 1, 1009, 61312, 32, 8, 128, name="resident_extend_1009_over_61312", causal=True),
        # One decoding step: a query for each of 24 sequences of 8,000 keys on
        # average.
        _case("resident", 24, 24, 192007, 32, 8, 128, name="resident_decode24_gqa", causal=True, ragged=True),
        # Wide heads, an odd length.
        _case("resident", 1, 8190, 8190, 16, 16, 256, name="resident_8190x16_d256_causal", causal=True),
        # The benchmark's 65,536 x 32 x 128, resident in HBM.
        _case("resident", 1, 65536, 65536, 32, 32, 128, name="resident_65536x32_d128"),
        # A long causal prefill with the headline's 56 query heads.
        _case("resident", 1, 32768, 32768, 56, 8, 128, name="resident_32768x56_causal_gqa", causal=True),
        # The functional API on host tensors: 4,096 tokens, 8 heads of 64.
        _case("host", 2, 2 * 4096, 2 * 4096, 8, 8, 64, name="host_func_batch2_4096x8_d64", entry="func"),
        # The benchmark's streamed workload: pinned DRAM to pinned DRAM, 1 GiB
        # of workspace, head groups.
        _case("host", 1, 65536, 65536, 32, 32, 128, name="host_head_groups_65536x32_1gib", schedule="head_groups",
              budget_mib=1024, kv_chunk=4096),
        # INT8 K/V in three chunks applied to a resident block of queries.
        _case("chunks", 1, 6144, 3 * 8192, 32, 8, 128, name="chunks_int8_6144_over_3x8192", kv_chunk=8192, int8=True,
              outliers=True),
        # Pages of 256 tokens, 1% outlier keys, output left in HBM.
        _case("paged", 1, 16384, 16384, 16, 16, 128, name="paged_16384x16_d128", budget_mib=1024, page=256,
              outliers=True),
    ]


def _size(rng, low, high):
    """A size spread over the logarithm of [low, high], mostly odd ones."""
    n = int(round(low * (high / low) ** rng.random()))
    return max(low, n // 64 * 64) if rng.random() < 0.3 else n


def draw(rng: random.Random):
    """One more case of the listed kinds, with at most the largest listed one's work."""
    kind = rng.choice(["resident"] * 7 + ["host"] * 2 + ["chunks"] * 2 + ["paged"])
    dtype = rng.choice(["bf16", "bf16", "fp16"])
    causal = rng.random() < 0.5
    outliers = rng.random() < 0.25
    q_heads, kv_heads = rng.choice([(8, 8), (16, 16), (32, 32), (32, 8), (40, 8), (12, 4), (8, 2), (56, 8), (28, 4)])
    head_dim = rng.choice([64, 64, 128, 128, 128, 96, 80, 256])
    if kind == "resident":
        form = rng.choice(["one", "one", "batch", "ragged", "extend", "decode"])
        if form == "decode":
            segments = rng.randint(1, 48)
            return _case(kind, segments, segments, max(_size(rng, 4096, 400_000), segments), q_heads, kv_heads,
                         head_dim, dtype=dtype, causal=True, ragged=True, outliers=outliers)
        if form == "extend":
            kv = _size(rng, 4096, 131_072)
            return _case(kind, 1, _size(rng, 2, min(4096, kv // 2)), kv, q_heads, kv_heads, head_dim, dtype=dtype,
                         causal=causal, outliers=outliers)
        if form == "one":
            n = _size(rng, 100, 40_000)
            return _case(kind, 1, n, n, q_heads, kv_heads, head_dim, dtype=dtype, causal=causal, outliers=outliers)
        segments = rng.randint(2, 32)
        n = _size(rng, 64, 3000) * segments
        return _case(kind, segments, n, n, q_heads, kv_heads, head_dim, dtype=dtype, causal=causal,
                     ragged=form == "ragged", outliers=outliers)
    if kind == "host":
        if rng.random() < 0.5:
            segments = rng.randint(1, 4)
            n = _size(rng, 256, 6000) * segments
            return _case(kind, segments, n, n, q_heads, kv_heads, head_dim, dtype=dtype, causal=causal,
                         outliers=outliers, entry="func")
        n = _size(rng, 2048, 24_000)
        return _case(kind, 1, n, n, q_heads, kv_heads, head_dim, dtype=dtype, causal=causal, outliers=outliers,
                     schedule=rng.choice(["q_blocks", "head_groups"]), budget_mib=1024)
    if kind == "chunks":
        int8 = rng.random() < 0.5
        chunk = rng.choice([1024, 4096, 8192])
        return _case(kind, 1, _size(rng, 64, 12_000), chunk * rng.randint(1, 3) + rng.randint(0, 500), q_heads,
                     kv_heads, rng.choice([64, 128]) if int8 else head_dim, dtype=dtype, causal=False,
                     outliers=outliers, kv_chunk=chunk, int8=int8)
    n = _size(rng, 2000, 16_000)
    return _case(kind, 1, n, n, q_heads, kv_heads, rng.choice([64, 128]), dtype=dtype, causal=causal,
                 outliers=outliers, budget_mib=1024, page=256)


def _split(total, parts, ragged, fixed):
    """Lengths of `parts` segments that add up to `total`; ragged ones are the same for every seed."""
    if not ragged:
        return [total // parts + (1 if i < total % parts else 0) for i in range(parts)]
    rng = random.Random(fixed)
    weights = [rng.uniform(0.2, 1.8) for _ in range(parts)]
    lengths = [max(1, int(total * w / sum(weights))) for w in weights]
    while sum(lengths) > total:
        lengths[lengths.index(max(lengths))] -= 1
    lengths[-1] += total - sum(lengths)
    return lengths


def _lengths(case):
    """(query lengths, key lengths) of the case's segments."""
    k = _split(case["kv_tokens"], case["segments"], case["ragged"], case["segments"])
    if case["q_tokens"] == case["kv_tokens"]:
        return list(k), k
    return _split(case["q_tokens"], case["segments"], False, 0), k


def _bounds(lengths):
    return [0, *itertools.accumulate(lengths)]


def _inputs(case, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    dtype = DTYPES[case["dtype"]]

    def normal(tokens, heads):
        out = torch.empty((tokens, heads, case["head_dim"]), dtype=dtype, device="cuda")
        for start in range(0, tokens, 16384):  # in pieces: few temporaries
            rows = out[start : start + 16384]
            rows.copy_(torch.randn(rows.shape, generator=gen, device="cuda"))
        return out

    q, k, v = (normal(case["q_tokens"], case["q_heads"]), normal(case["kv_tokens"], case["kv_heads"]),
               normal(case["kv_tokens"], case["kv_heads"]))
    if case["outliers"]:
        rows = torch.randperm(case["kv_tokens"], generator=gen, device="cuda")[: max(1, case["kv_tokens"] // 100)]
        k[rows] *= 8
    return q, k, v


def _quantized(x):
    """INT8 rows and one fp16 scale per 64 tokens and head, as the INT8 pages hold them."""
    tokens, heads, dim = x.shape
    groups = -(-tokens // QUANT_GROUP)
    padded = torch.zeros((groups * QUANT_GROUP, heads, dim), dtype=torch.float32, device=x.device)
    padded[:tokens] = x.float()
    grouped = padded.view(groups, QUANT_GROUP, heads, dim)
    step = grouped.abs().amax(dim=(1, 3)) / 127.0
    step = torch.where(step > 0, step, torch.ones_like(step))
    q8 = torch.round(grouped / step[:, None, :, None]).clamp_(-127, 127).to(torch.int8)
    return q8.view(groups * QUANT_GROUP, heads, dim)[:tokens].contiguous(), step.to(torch.float16)


def _pinned(x):
    host = torch.empty(x.shape, dtype=x.dtype, pin_memory=True)
    host.copy_(x)
    return host


def _config(case):
    return seqattn.StreamingAttentionConfig(
        workspace_budget_bytes=case["budget_mib"] * 2**20 or None, kv_chunk_tokens=case["kv_chunk"] or None,
        schedule=case["schedule"],
    )


def _plan(case, config):
    return seqattn.build_plan(
        q_heads=case["q_heads"], kv_heads=case["kv_heads"], head_dim=case["head_dim"], dtype=DTYPES[case["dtype"]],
        device="cuda", max_q_tokens=case["q_tokens"], max_kv_tokens=case["kv_tokens"], config=config,
    )


def prepare(case, seed):
    q, k, v = _inputs(case, seed)
    q_lengths, k_lengths = _lengths(case)
    state = {"case": case, "cu_q": torch.tensor(_bounds(q_lengths), dtype=torch.int32),
             "cu_k": torch.tensor(_bounds(k_lengths), dtype=torch.int32)}
    kind = case["kind"]
    if kind == "resident":
        config = _config(case)
        state.update(q=q, k=k, v=v, runner=seqattn.StreamingAttentionRunner(_plan(case, config), config))
    elif kind == "host":
        q, k, v = _pinned(q), _pinned(k), _pinned(v)
        if case["entry"] == "func":
            batch = case["segments"]
            state.update(q=q.unflatten(0, (batch, -1)), k=k.unflatten(0, (batch, -1)), v=v.unflatten(0, (batch, -1)))
        else:
            config = _config(case)
            state.update(q=q, k=k, v=v, out=torch.empty(q.shape, dtype=q.dtype, pin_memory=True),
                         lse=torch.empty((case["q_heads"], case["q_tokens"]), device="cuda"),
                         runner=seqattn.StreamingAttentionRunner(_plan(case, config), config))
    elif kind == "chunks":
        rows, heads, dim = q.shape
        state.update(q=q, k=k, v=v, m=torch.empty((rows, heads), device="cuda"),
                     l=torch.empty((rows, heads), device="cuda"), acc=torch.empty((rows, heads, dim), device="cuda"),
                     out=torch.empty_like(q), lse=torch.empty((heads, rows), device="cuda"))
        if case["int8"]:
            state["k"], state["k_scales"] = _quantized(k)
            state["v"], state["v_scales"] = _quantized(v)
    else:
        q, k, v = _pinned(q), _pinned(k), _pinned(v)
        page_bytes = case["page"] * case["kv_heads"] * case["head_dim"] * 2
        source = seqattn.MemoryPageSource(q=q, k=k, v=v, cu_seqlens_q=state["cu_q"], cu_seqlens_k=state["cu_k"],
                                          page_target_bytes=page_bytes, block_n=64)
        config = seqattn.PagedAttentionConfig(
            attention=seqattn.StreamingAttentionConfig(workspace_budget_bytes=case["budget_mib"] * 2**20),
            page_target_bytes=page_bytes, kv_storage_dtype=case["dtype"],
        )
        state.update(source=source, runner=seqattn.PagedAttentionRunner(config),
                     out=torch.empty(q.shape, dtype=q.dtype, device="cuda"),
                     lse=torch.empty((case["q_heads"], case["q_tokens"]), device="cuda"))
    return state


def _run_chunks(state):
    case = state["case"]
    q, k, v = state["q"], state["k"], state["v"]
    total = case["kv_tokens"]
    for start in range(0, total, case["kv_chunk"]):
        stop = min(start + case["kv_chunk"], total)
        common = dict(q_tokens=q.shape[0], kv_tokens=stop - start, q_local_offset=0, kv_local_offset=start,
                      causal_shift=total - q.shape[0], softmax_scale=case["head_dim"] ** -0.5, causal=case["causal"],
                      initialize=start == 0)
        if case["int8"]:
            update_attention_state_int8(q, k[start:stop], v[start:stop], state["k_scales"], state["v_scales"],
                                        state["m"], state["l"], state["acc"], storage_token_offset=start, **common)
        else:
            update_attention_state(q, k[start:stop], v[start:stop], state["m"], state["l"], state["acc"], **common)
    finalize_attention(state["acc"], state["l"], state["out"], q_tokens=q.shape[0], running_max=state["m"],
                       lse=state["lse"])
    return state["out"], state["lse"]


def run(state):
    case = state["case"]
    kind = case["kind"]
    if kind == "resident":
        return state["runner"](state["q"], state["k"], state["v"], state["cu_q"], state["cu_k"],
                               causal=case["causal"], return_lse=True)
    if kind == "host":
        if case["entry"] == "func":
            return seqattn.streaming_attn_func(state["q"], state["k"], state["v"], causal=case["causal"])
        return state["runner"](state["q"], state["k"], state["v"], state["cu_q"], state["cu_k"],
                               causal=case["causal"], out=state["out"], lse_out=state["lse"], return_lse=True)
    if kind == "chunks":
        return _run_chunks(state)
    out = state["runner"].run_with_device_output(state["source"], state["source"], state["cu_q"], state["cu_k"],
                                                 out=state["out"], causal=case["causal"], lse_out=state["lse"])
    return out, state["lse"]


def _pairs(case):
    """Visible (query, key) pairs of one head, bottom-right causal."""
    pairs = 0
    for n_q, n_k in zip(*_lengths(case)):
        if not case["causal"]:
            pairs += n_q * n_k
            continue
        first = n_k - n_q + 1  # keys the first query sees
        hidden = max(0, -(n_k - n_q))  # leading queries that see none
        pairs += (n_q - hidden) * (max(first, 1) + n_k) // 2
    return pairs


def work(case):
    kv_bytes = 2 * case["kv_tokens"] * case["kv_heads"] * case["head_dim"] * (1 if case["int8"] else 2)
    if case["int8"]:
        kv_bytes += 2 * 2 * case["kv_heads"] * -(-case["kv_tokens"] // QUANT_GROUP)
    q_bytes = case["q_tokens"] * case["q_heads"] * case["head_dim"] * 2
    lse_bytes = case["q_tokens"] * case["q_heads"] * 4
    return {"bytes": kv_bytes + 2 * q_bytes + lse_bytes,
            "flops": 4 * case["head_dim"] * case["q_heads"] * _pairs(case)}


def tolerance(case):
    # Four times the distance from 64 bits that the path shows: P and the
    # output are rounded to the 16-bit type (bf16 2.3e-3, fp16 2.9e-4); INT8
    # K/V are rounded to it too, after their scale.
    if case["int8"]:
        return {"rel": 2e-2 if case["dtype"] == "bf16" else 3e-3}
    return {"rel": 1e-2 if case["dtype"] == "bf16" else 1.2e-3}


def exact(case, seed):
    q, k, v = _inputs(case, seed)
    if case["int8"]:
        k, v = (q8.double() * scales.double().repeat_interleave(QUANT_GROUP, dim=0)[: q8.shape[0], :, None]
                for q8, scales in (_quantized(k), _quantized(v)))
    heads, dim = q.shape[1:]
    group = heads // k.shape[1]
    out = torch.empty(q.shape, dtype=torch.float64, device="cuda")
    lse = torch.empty((heads, q.shape[0]), dtype=torch.float64, device="cuda")
    q_lengths, k_lengths = _lengths(case)
    for q0, q1, k0, k1 in zip(_bounds(q_lengths), _bounds(q_lengths)[1:], _bounds(k_lengths), _bounds(k_lengths)[1:]):
        shift = (k1 - k0) - (q1 - q0)
        rows = max(1, 2**28 // (k1 - k0))
        keys = torch.arange(k1 - k0, device="cuda")
        for head in range(heads):
            kd, vd = k[k0:k1, head // group].double(), v[k0:k1, head // group].double()
            for start in range(q0, q1, rows):
                stop = min(start + rows, q1)
                s = (q[start:stop, head].double() * dim**-0.5) @ kd.T.contiguous()
                if case["causal"]:
                    seen = torch.arange(start - q0, stop - q0, device="cuda") + shift
                    s.masked_fill_(keys[None, :] > seen[:, None], float("-inf"))
                top = s.amax(dim=1, keepdim=True).clamp_min_(-1e300)
                s.sub_(top).exp_()
                total = s.sum(dim=1, keepdim=True)
                lse[head, start:stop] = (top + total.log())[:, 0]
                out[start:stop, head] = (s @ vd) / total.clamp_min(1e-300)
    if case["entry"] == "func":
        return out.unflatten(0, (case["segments"], -1))
    return out, lse
