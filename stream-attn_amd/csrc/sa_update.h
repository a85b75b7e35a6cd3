// The chunk-update kernel of the streamed exact-attention path for MI355X
// (gfx950, CDNA4), as a template over its geometry, and the launch of one
// variant.  sa_kernels.hip chooses the variant; each head-dim's variants are
// compiled in a source file of their own (sa_update_d*.hip).
//
// Semantics follow _streaming_attention_update_kernel (reference
// src/seqattn_core/kernels/streaming.py:19-156): base-2 online softmax over
// one K/V chunk, FP32 state (m, l, acc) carried in HBM between chunks, P
// rounded to the input dtype before the PV product.
//
// Work decomposition: a workgroup is 8 wavefronts (two per SIMD), each owning
// QB 16-query blocks of one query head as 16x16x32 MFMAs, 128 QB queries per
// workgroup; while one wave of a SIMD waits on LDS or on the MFMA pipe the
// other issues.  Each K/V fragment read from LDS feeds QB MFMAs.
// K/V stream through LDS in 64-key tiles, two stages: the tile after the one
// being computed is fetched by global_load_lds_dwordx4 (HBM/L2 -> LDS with
// no register staging) while the MFMAs run; one barrier per tile.  Small
// launches over many keys have four stages, three tiles in flight
// (choose_stages).
//
// v_mfma_f32_16x16x32_{bf16,f16}: A 16x32 (lane l: row l % 16, k 8 (l / 16)
// .. +7), B 32x16 (lane l: column l % 16, k 8 (l / 16) .. +7), C 16x16 (lane
// l: column l % 16, rows 4 (l / 16) .. +3).  With j = l / 16:
//   S^T[key][query] = K . Q^T: A = K rows (LDS), B = Q (registers for the
//   whole kernel).  The lane holds query l % 16 of each block and keys
//   4j .. 4j + 3 of each 16-key block of the 32-key step.
//   O^T[d][query] += V^T . P^T: B = P^T straight from those registers, k slot
//   8j + e holding key 4j + e (e < 4) or 16 + 4j + e - 4; A = V^T rows in
//   the same slot order, from two transposing LDS reads per fragment (or one
//   16-byte read of the transposed copy of V).
// A query's 32 keys of a step are spread over four lanes (j = 0..3); its
// partial row sums stay per lane and are added in the fixed order
// (l0 + l1) + (l2 + l3) wherever l is stored or merged.
//
// Online softmax with a thresholded rescale: a query's running maximum m only
// moves (and its acc, l are rescaled by exp2(m_old - m_new)) when one of its
// logits exceeds m + 8; otherwise p = exp2(s*scale - m) <= 2^8 against the
// kept m.  The decision is per query, so results do not depend on how queries
// are grouped into wavefronts, workgroups or Q blocks: every QB gives the
// same bits.
// Each step first computes P against the kept m and tests the lane's partial
// row sum: every p <= 2^8 whenever that sum is, so the row maximum (and its
// cross-lane exchange) is only taken on the rare steps that may rescale, and
// the result is the same as deciding on the maximum.
// (m, l, acc) remains an exact representation of the partial softmax:
// out = acc / l and LSE = m + log2(l) are unchanged, and P keeps bf16's
// relative precision.
//
// INT8 K/V (update_attention_state_int8, reference kernels/streaming.py:113-120
// and :274-342): int8 rows with one fp16 scale per (token group, K/V head).
// Raw int8 tiles (half the bytes of bf16) arrive by LDS DMA into a staging
// area; one pass per tile turns them into the bf16/fp16 stage layout as
// dtype(fp32(k) * fp32(scale)), exactly the reference's dequantization, so
// the MFMA loop is shared and the result equals the 16-bit kernel run on
// dequantized K/V bit for bit.  Per tile: DMA of tile t+2, dequantization of
// tile t+1 and the MFMAs of tile t, one barrier.  Each thread's scales for
// the next tile are loaded into registers one tile ahead.
#pragma once

#include <hip/hip_runtime.h>

#include <cstdint>

#include "sa_common.h"
#include "seqattn_hip.h"

namespace sa {

// How K and V arrive: 16-bit rows, 16-bit K rows with V transposed per K/V
// head, INT8 rows with scales.
enum KVMode { kRows = 0, kTransposedV = 1, kInt8 = 2 };

// How workgroups are numbered (hardware block b runs on XCD b % 8).
enum Numbering {
  // Each XCD takes an eighth of the heads of every segment, so the
  // workgroups resident on one XCD share few heads' K/V in its L2.
  kHeadsPerXcd = 0,
  // Each XCD takes a contiguous eighth of the workgroups: one segment without
  // a mask whose heads are no multiple of 8.
  kRunsPerXcd = 1,
  // Consecutive workgroups go to consecutive XCDs: workgroups of unequal
  // length (a causal mask, segments) whose heads are no multiple of 8, of
  // which a contiguous run would give some XCD more than its share of long
  // ones (measured: 1.7x the runs' rate on one causal head, 1.14x on 12).
  kDealt = 2,
};

// Segments of one launch: the table travels in the kernel's arguments.
constexpr int kMaxSegments = 32;

struct UpdateParams {
  const uint16_t* q;
  const uint16_t* k;
  const uint16_t* v;
  float* m;
  float* l;
  float* acc;
  int64_t sq_t, sq_h, sk_t, sk_h, sv_t, sv_h, ss_t, ss_h, sa_t, sa_h;
  int32_t q_tokens, kv_tokens, group, head_dim, q_heads;
  int32_t q_local_offset, kv_local_offset, causal_shift;
  int32_t causal, init;
  // With pack (128-query workgroups of grouped-query launches) a row of a
  // workgroup is one (query, query head of the K/V head) pair, `group` pairs
  // per query, and unit_heads the K/V heads; else a row is a query and
  // unit_heads the query heads.
  int32_t pack, unit_heads;
  int32_t numbering;      // Numbering
  int32_t slots;          // workgroups of the launch (of one XCD, for kHeadsPerXcd)
  int32_t xcd_run;        // kRunsPerXcd: ceil(slots / 8)
  float scale_log2;
  // INT8 K/V only: fp16 scales, element (group, kv_head) at
  // scales[group * s?s_g + kv_head * s?s_h], group = (scale_offset + key) >> scale_shift.
  const uint16_t* ks;
  const uint16_t* vs;
  int64_t sks_g, sks_h, svs_g, svs_h;
  int32_t scale_offset, scale_shift;
  // 16-bit launches spanning several K/V chunks of the streamed schedule:
  // the tile count of one chunk (0: one chunk).  At each chunk boundary the
  // lanes' partial row sums are merged exactly as a chunk launch stores l and
  // the next one reloads it, so the result equals the chunked schedule's bit
  // for bit.
  int32_t merge_tiles;
  // Fused finalize, for the launch that applies the last keys of its rows
  // (with or without loading the state first): when out is non-null the
  // epilogue writes acc / l (0 where l == 0) to out and, when lse is
  // non-null, (m + log2 l) ln 2 (-inf where l == 0) to
  // lse[head * lse_sh + lse_off + query], with the expressions of
  // finalize_kernel, and stores no state.  out may alias q: what a wave uses
  // of a query's row of one head it reads at the start, and only that wave
  // writes the row, at the end.  (Lanes past the last query read the last
  // query's row too, possibly while it is being written, and drop the value.)
  uint16_t* out;
  int64_t so_t, so_h;
  float* lse;
  int64_t lse_sh, lse_off;
  // State in the pipeline's row-group layout (state_block) instead of the
  // strided [token][head] layout given by ss_* / sa_*.
  int32_t tiled_state;
  // With segments > 1 the launch covers that many, instead of q_tokens
  // queries over kv_tokens keys: their rows as in sa::Segment, and the first
  // workgroup number (see slots) of each.
  int32_t segments;
  int32_t first[kMaxSegments];
  Segment segment[kMaxSegments];
};

constexpr int kTileKeys = 64;
constexpr int kThreads = 512;       // of a workgroup: 8 waves
constexpr int kRowsPerBlock = 128;  // a workgroup's rows per 16-query block of its waves

// The compiled variants of a padded head_dim: queries per workgroup (8 waves
// of rows / 8), and the measured nanoseconds per 64-key tile of a workgroup
// alone on its CU (`one`) and of two workgroups sharing a CU (`two`, 0 where
// registers or LDS hold one): bf16, V read in place, 256 CUs busy.  The present
// build on another box takes 4-16% less throughout; with those figures 58 drawn
// launches choose the same widths.  (Up to four head_dim-32 workgroups fit on a
// CU; the model counts two.)
struct UpdateVariant {
  int32_t rows, one, two;
};
constexpr int kHeadDims = 4;  // 32, 64, 128, 256
constexpr int kMaxVariants = 3;
constexpr UpdateVariant kVariants[kHeadDims][kMaxVariants] = {
    {{128, 605, 920}, {256, 930, 1550}, {0, 0, 0}},
    {{128, 800, 1245}, {256, 1245, 2070}, {0, 0, 0}},
    {{128, 1265, 2025}, {256, 1915, 0}, {384, 2600, 0}},
    {{128, 2460, 0}, {256, 3505, 0}, {0, 0, 0}},
};

// Rows of a workgroup (a variant's), LDS stages (4 only with 128 rows, V read
// in place and head_dim up to 128) and workgroups of a launch.
struct LaunchShape {
  int32_t rows, stages;
  uint32_t grid;
};

// One launch with the head-dim's variant of that shape.
hipError_t launch_update_d32(const UpdateParams&, int mode, const LaunchShape&, int dtype, hipStream_t);
hipError_t launch_update_d64(const UpdateParams&, int mode, const LaunchShape&, int dtype, hipStream_t);
hipError_t launch_update_d128(const UpdateParams&, int mode, const LaunchShape&, int dtype, hipStream_t);
hipError_t launch_update_d256(const UpdateParams&, int mode, const LaunchShape&, int dtype, hipStream_t);

}  // namespace sa
