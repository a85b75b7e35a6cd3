// Device code of the chunk-update kernel (see sa_update.h) and its launch;
// included by the sources that compile one head-dim's variants.
#pragma once

#include <cmath>
#include <type_traits>

#include "sa_update.h"

namespace sa {
namespace {

typedef uint32_t u32x4 __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2 __attribute__((ext_vector_type(2)));
typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef _Float16 f16x8 __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x2 __attribute__((ext_vector_type(2)));
typedef _Float16 f16x2 __attribute__((ext_vector_type(2)));

#define SA_LDS __attribute__((address_space(3)))
#define SA_GLOBAL __attribute__((address_space(1)))
#define SA_CONSTANT __attribute__((address_space(4)))

constexpr int kSubKeys = 32;   // keys per softmax step
constexpr float kRescaleThreshold = 8.0f;  // log2 units

struct BF16 {
  __device__ static inline f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8, a), __builtin_bit_cast(bf16x8, b), c,
                                                   0, 0, 0);
  }
  // Two floats -> two round-to-nearest-even bf16 packed in one dword (low = a).
  __device__ static inline uint32_t pack2(float a, float b) {
    bf16x2 v = {(__bf16)a, (__bf16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
};

struct FP16 {
  __device__ static inline f32x4 mma(u32x4 a, u32x4 b, f32x4 c) {
    return __builtin_amdgcn_mfma_f32_16x16x32_f16(__builtin_bit_cast(f16x8, a), __builtin_bit_cast(f16x8, b), c,
                                                  0, 0, 0);
  }
  __device__ static inline uint32_t pack2(float a, float b) {
    f16x2 v = {(_Float16)a, (_Float16)b};
    return __builtin_bit_cast(uint32_t, v);
  }
};

// Pipeline-owned FP32 state is kept in the order the update kernel's lanes
// hold it.  Rows form groups of 16; group g of head h is one block of
// 16 * head_dim floats (and 16 floats of m, of l) at block index
// g * q_heads + h, so row r of a buffer sits where the token-major layout
// would put it, rounded to its 16-row group.  Within a block, 4-float chunk c
// (d = 4c .. 4c + 3) of row r is at (c * 16 + r) * 4.  The 64 lanes' chunks
// of one 16-wide d block are then 1 KB of contiguous memory, where the
// token-major layout touched one 16-byte piece per row, rows
// q_heads * head_dim * 4 bytes apart.
__device__ inline int64_t state_block(int64_t row, int head, int q_heads) {
  return (row >> 4) * q_heads + head;
}

// Positive factor applied to raw logits inside the exponent's FMA (so the
// running max can be taken before scaling): |scale|, at least 1e-30.
__device__ inline float scale_factor(float scale_log2) { return fmaxf(fabsf(scale_log2), 1e-30f); }

// Sign-bit mask that negates every 16-bit element of a Q fragment when the
// scale is negative: s * scale == (-q . k) * |scale|, exactly.
__device__ inline u32x4 q_sign(float scale_log2) {
  const uint32_t m = scale_log2 < 0.f ? 0x80008000u : 0u;
  return u32x4{m, m, m, m};
}

// Fragment reads from LDS.  A batch's reads and the wait for them are one asm
// statement: the compiler takes an asm's outputs as written when it ends, so a
// read whose wait stood in a later statement could be copied or overwritten
// while in flight.  The outputs are early-clobber (later reads of the batch
// still need the address).  asm rather than plain loads because the compiler
// cannot relate an LDS read to the DMA writing the other stage and would wait
// for that prefetch (vmcnt) before it, and because its own schedule waited
// three times per step (with the second wave of the SIMD usually waiting at
// the same moment); plain loads and the transposing builtin at head_dim 256
// took 2-14% more.

// w[kb N / 2 + c] = the 16 bytes at addr + base + kb * step + c KB.
template <int N>
__device__ inline __attribute__((always_inline)) void read_k(u32x4 (&w)[N], uint32_t addr, int base, int step) {
  static_assert(N == 2 || N == 4 || N == 8, "K fragments of a batch");
  if constexpr (N == 2)
    asm volatile(
        "ds_read_b128 %0, %2 offset:%3\n\t"
        "ds_read_b128 %1, %2 offset:%3+%4\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]) : "v"(addr), "i"(base), "i"(step) : "memory");
  else if constexpr (N == 4)
    asm volatile(
        "ds_read_b128 %0, %4 offset:%5\n\t"
        "ds_read_b128 %2, %4 offset:%5+%6\n\t"
        "ds_read_b128 %1, %4 offset:%5+1024\n\t"
        "ds_read_b128 %3, %4 offset:%5+%6+1024\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]) : "v"(addr), "i"(base), "i"(step) : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %8 offset:%9\n\t"
        "ds_read_b128 %4, %8 offset:%9+%10\n\t"
        "ds_read_b128 %1, %8 offset:%9+1024\n\t"
        "ds_read_b128 %5, %8 offset:%9+%10+1024\n\t"
        "ds_read_b128 %2, %8 offset:%9+2048\n\t"
        "ds_read_b128 %6, %8 offset:%9+%10+2048\n\t"
        "ds_read_b128 %3, %8 offset:%9+3072\n\t"
        "ds_read_b128 %7, %8 offset:%9+%10+3072\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7])
        : "v"(addr), "i"(base), "i"(step)
        : "memory");
}

// w[dd] = the 16 bytes at addr + base + dd KB.
template <int N>
__device__ inline __attribute__((always_inline)) void read_vt(u32x4 (&w)[N], uint32_t addr, int base) {
  static_assert(N == 4 || N == 8, "V^T fragments of a batch");
  if constexpr (N == 4)
    asm volatile(
        "ds_read_b128 %0, %4 offset:%5\n\t"
        "ds_read_b128 %1, %4 offset:%5+1024\n\t"
        "ds_read_b128 %2, %4 offset:%5+2048\n\t"
        "ds_read_b128 %3, %4 offset:%5+3072\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]) : "v"(addr), "i"(base) : "memory");
  else
    asm volatile(
        "ds_read_b128 %0, %8 offset:%9\n\t"
        "ds_read_b128 %1, %8 offset:%9+1024\n\t"
        "ds_read_b128 %2, %8 offset:%9+2048\n\t"
        "ds_read_b128 %3, %8 offset:%9+3072\n\t"
        "ds_read_b128 %4, %8 offset:%9+4096\n\t"
        "ds_read_b128 %5, %8 offset:%9+5120\n\t"
        "ds_read_b128 %6, %8 offset:%9+6144\n\t"
        "ds_read_b128 %7, %8 offset:%9+7168\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(w[0]), "=&v"(w[1]), "=&v"(w[2]), "=&v"(w[3]), "=&v"(w[4]), "=&v"(w[5]), "=&v"(w[6]), "=&v"(w[7])
        : "v"(addr), "i"(base)
        : "memory");
}

// w[dd]: d block dd of the batch (an even one first) from V's rows, its two
// 16-key blocks 1 KB apart, each pair of d blocks 4 KB from the next; the odd
// block of a pair is read at addr_odd.
template <int N>
__device__ inline __attribute__((always_inline)) void read_v(u32x4 (&w)[N], uint32_t addr, uint32_t addr_odd, int base) {
  static_assert(N == 2 || N == 4 || N == 8, "V fragments of a batch");
  u32x2 h[2 * N];
  if constexpr (N == 2)
    asm volatile(
        "ds_read_b64_tr_b16 %0, %4 offset:%6\n\t"
        "ds_read_b64_tr_b16 %1, %4 offset:%6+1024\n\t"
        "ds_read_b64_tr_b16 %2, %5 offset:%6\n\t"
        "ds_read_b64_tr_b16 %3, %5 offset:%6+1024\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]) : "v"(addr), "v"(addr_odd), "i"(base) : "memory");
  else if constexpr (N == 4)
    asm volatile(
        "ds_read_b64_tr_b16 %0, %8 offset:%10\n\t"
        "ds_read_b64_tr_b16 %1, %8 offset:%10+1024\n\t"
        "ds_read_b64_tr_b16 %2, %9 offset:%10\n\t"
        "ds_read_b64_tr_b16 %3, %9 offset:%10+1024\n\t"
        "ds_read_b64_tr_b16 %4, %8 offset:%10+4096\n\t"
        "ds_read_b64_tr_b16 %5, %8 offset:%10+5120\n\t"
        "ds_read_b64_tr_b16 %6, %9 offset:%10+4096\n\t"
        "ds_read_b64_tr_b16 %7, %9 offset:%10+5120\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(h[4]), "=&v"(h[5]), "=&v"(h[6]), "=&v"(h[7])
        : "v"(addr), "v"(addr_odd), "i"(base)
        : "memory");
  else
    asm volatile(
        "ds_read_b64_tr_b16 %0, %16 offset:%18\n\t"
        "ds_read_b64_tr_b16 %1, %16 offset:%18+1024\n\t"
        "ds_read_b64_tr_b16 %2, %17 offset:%18\n\t"
        "ds_read_b64_tr_b16 %3, %17 offset:%18+1024\n\t"
        "ds_read_b64_tr_b16 %4, %16 offset:%18+4096\n\t"
        "ds_read_b64_tr_b16 %5, %16 offset:%18+5120\n\t"
        "ds_read_b64_tr_b16 %6, %17 offset:%18+4096\n\t"
        "ds_read_b64_tr_b16 %7, %17 offset:%18+5120\n\t"
        "ds_read_b64_tr_b16 %8, %16 offset:%18+8192\n\t"
        "ds_read_b64_tr_b16 %9, %16 offset:%18+9216\n\t"
        "ds_read_b64_tr_b16 %10, %17 offset:%18+8192\n\t"
        "ds_read_b64_tr_b16 %11, %17 offset:%18+9216\n\t"
        "ds_read_b64_tr_b16 %12, %16 offset:%18+12288\n\t"
        "ds_read_b64_tr_b16 %13, %16 offset:%18+13312\n\t"
        "ds_read_b64_tr_b16 %14, %17 offset:%18+12288\n\t"
        "ds_read_b64_tr_b16 %15, %17 offset:%18+13312\n\t"
        "s_waitcnt lgkmcnt(0)"
        : "=&v"(h[0]), "=&v"(h[1]), "=&v"(h[2]), "=&v"(h[3]), "=&v"(h[4]), "=&v"(h[5]), "=&v"(h[6]), "=&v"(h[7]),
          "=&v"(h[8]), "=&v"(h[9]), "=&v"(h[10]), "=&v"(h[11]), "=&v"(h[12]), "=&v"(h[13]), "=&v"(h[14]), "=&v"(h[15])
        : "v"(addr), "v"(addr_odd), "i"(base)
        : "memory");
#pragma unroll
  for (int dd = 0; dd < N; ++dd) w[dd] = u32x4{h[2 * dd][0], h[2 * dd][1], h[2 * dd + 1][0], h[2 * dd + 1][1]};
}

// DP: head_dim padded to 32, 64, 128 or 256.
template <int DP>
struct Geometry {
  static constexpr int WAVES = 8;
  static constexpr int THREADS = 64 * WAVES;
  static constexpr int CK = DP / 32;                           // 32-wide d steps of QK^T
  static constexpr int DB = DP / 16;                           // 16-wide d blocks of the output
  static constexpr int TILE_BYTES = kTileKeys * DP * 2;        // K (or V) part of a stage
  static constexpr int PIECES = TILE_BYTES / 1024;             // wave-wide DMAs of one tensor's tile
  // Waves 0-3 (the first wave of each SIMD) issue the tile DMA.
  static constexpr int ISSUERS = 4;
  static constexpr int I8_TILE_BYTES = kTileKeys * DP;
  static constexpr int I8_GR = DP / 16;                        // 16-byte granules per int8 row
  static constexpr int I8_DMAS = I8_TILE_BYTES / 1024;
  static constexpr int I8_GRANULES = kTileKeys * I8_GR;
  static_assert(PIECES % ISSUERS == 0 && WAVES >= ISSUERS, "tile geometry");
  // LDS layouts of one stage.  A wave-wide DMA writes 1 KB of LDS linearly,
  // 16 bytes per lane, so the layouts keep 64 bytes of one global row in four
  // consecutive lanes (one cache request) and permute the 16-byte granules
  // within them so that every fragment read below is free of bank conflicts.
  // Every fragment read is a per-lane base plus a compile-time offset (the
  // instruction's immediate).
  //   K: the 16-key x 32-d A fragment (16-key block kb, d block c) is 1 KB at
  //   (CK kb + c) KB, 64 bytes per key, granule g of the key's four at slot
  //   k_slot(g) ^ (key / 4 % 4).  A ds_read_b128 serves lanes 0-3, 12-15 and
  //   20-27 of each half wave in one cycle and the others in the next; with
  //   k_slot = 0, 3, 1, 2 both sets of 16 touch every slot of 256 bytes once
  //   (with k_slot(g) = g every read took 4 more cycles).
  //   V: blocks of 32 d, 64 keys x 64 bytes each, granule g of a key's four
  //   at slot g ^ 2 (key / 4 % 2).  A transposing read has each 16-lane group
  //   take 32 bytes of 4 consecutive keys; two neighbouring groups use both
  //   halves of their 256 bytes.
  //   V^T (transposed copy, stored tile by tile in this order): the 16-d x
  //   32-key fragment (32-key block sb, d block db) at (DB sb + db) KB, lane
  //   (j, r16)'s 16 bytes (row 16 db + r16, key granule 4 sb + j) at 16 * lane.
  __device__ static inline int k_slot(int g) { return ((g & 1) << 1) | ((g ^ (g >> 1)) & 1); }
  __device__ static inline int k_granule(int slot) { return (((slot ^ (slot >> 1)) & 1) << 1) | (slot >> 1); }
  __device__ static inline int k_offset(int key, int g) {
    return ((key >> 4) * CK + (g >> 2)) * 1024 + (key & 15) * 64 + ((k_slot(g & 3) ^ ((key >> 2) & 3)) << 4);
  }
  __device__ static inline int v_offset(int key, int g) {
    return (g >> 2) * 4096 + key * 64 + (((g & 3) ^ (2 * ((key >> 2) & 1))) << 4);
  }
};

// V of kTransposedV: per K/V head a copy of V in the V^T layout above, 64-key
// tile by tile, each 32-key group in the k-slot order of P^T (slot s holds
// key 16 ((s >> 2) & 1) + 4 (s >> 3) + (s & 3)), zero keys up to a multiple
// of 64.
// STAGES: LDS stages, of which all but one are in flight while a tile is
// computed (2, or 4 for V read in place).
template <typename Op, int DP, int QB, int MODE, int STAGES>
__global__ __launch_bounds__(Geometry<DP>::THREADS) void update_kernel(const UpdateParams p) {
  using Geo = Geometry<DP>;
  constexpr bool VT = MODE == kTransposedV;
  constexpr bool QUANT = MODE == kInt8;
  constexpr bool RING = STAGES > 2;
  static_assert(STAGES == 2 || (STAGES == 4 && MODE == kRows), "LDS stages");
  constexpr int CK = Geo::CK;
  constexpr int DB = Geo::DB;
  // Fragments read before one wait: KB 32-wide d steps of K (two fragments
  // each) and VB d blocks of V, as many as the registers hold.  Measured:
  // head_dim 256, 32 queries per wave, 9,239 x 16 heads 1,350 us with (2, 4),
  // 1,379 with (2, 2) or (1, 4), more with spills above; 16 queries, 200 over
  // 20,000 keys x 16 heads 703 us with (4, 8), 722 with (4, 4), 735 with (2, 8).
  // head_dim 128, 48 queries per wave 2.45 us a tile on a full chip with VB 8,
  // 2.50 with 2; 16 queries, 1,009 over 61,312 keys x 32/8 heads 1,058 us with
  // (4, 4), 1,071 with (2, 4) or (4, 8), and with INT8 K/V, 667 over 8,446 keys
  // x 40/8 heads, 240 us with (2, 4), 243 with (4, 4), 249 with (4, 8).
  constexpr int KB = DP == 256 ? (QB == 1 ? 4 : 2) : DP == 128 && QUANT && QB == 1 ? 2 : CK;
  constexpr int VB = DP == 256 ? (QB == 1 ? 8 : 4) : DP == 32 ? 2 : DP == 128 && QB > 1 ? 8 : 4;
  constexpr int BLOCK_M = Geo::WAVES * 16 * QB;
  static_assert(!QUANT || (Geo::I8_DMAS <= Geo::WAVES && Geo::I8_GRANULES <= Geo::THREADS), "INT8 staging");

  // Two LDS stages as distinct objects: every LDS read and every DMA target
  // below names one of them statically, so the compiler can tell that the
  // in-flight prefetch into one stage does not alias reads of the other and
  // need not wait for it.
  // A ring of more stages is lds_a alone: its tiles are only read by inline
  // asm, which the compiler does not relate to the DMA (no wait of its own
  // stands in the loop).
  constexpr int STAGE_BYTES = 2 * Geo::TILE_BYTES;
  __shared__ __attribute__((aligned(1024))) uint8_t lds_a[RING ? STAGES * STAGE_BYTES : STAGE_BYTES];
  __shared__ __attribute__((aligned(1024))) uint8_t lds_b[RING ? 16 : STAGE_BYTES];
  // INT8 staging (K then V of one raw tile), also two distinct objects.
  constexpr int kStagingBytes = QUANT ? 2 * Geo::I8_TILE_BYTES : 16;
  __shared__ __attribute__((aligned(1024))) uint8_t lds_qa[kStagingBytes];
  __shared__ __attribute__((aligned(1024))) uint8_t lds_qb[kStagingBytes];

  const SA_CONSTANT UpdateParams* args = (const SA_CONSTANT UpdateParams*)__builtin_amdgcn_kernarg_segment_ptr();

  // Workgroup -> (segment, head, query block), numbered segment by segment
  // and head by head (see Numbering).  Under a causal mask later query blocks
  // see more keys: they come first so that the short blocks fill the end of
  // the launch.
  const int b = blockIdx.x;
  int slot = p.numbering == kDealt ? b : b >> 3;
  if (p.numbering == kRunsPerXcd) slot += (b & 7) * p.xcd_run;
  if (slot >= p.slots) return;
  int q_tokens = p.q_tokens, kv_tokens = p.kv_tokens, causal_shift = p.causal_shift;
  int q0 = 0, k0 = 0;
  if (p.segments > 1) {
    // Every lane looks at one segment's first number.
    const int at = threadIdx.x & 63;
    const bool before = at < p.segments && args->first[at & (kMaxSegments - 1)] <= slot;
    const int s = __builtin_amdgcn_readfirstlane(__popcll(__ballot(before)) - 1);
    slot -= __builtin_amdgcn_readfirstlane(args->first[s]);
    q0 = __builtin_amdgcn_readfirstlane(args->segment[s].q0);
    k0 = __builtin_amdgcn_readfirstlane(args->segment[s].k0);
    q_tokens = __builtin_amdgcn_readfirstlane(args->segment[s].q_len);
    kv_tokens = __builtin_amdgcn_readfirstlane(args->segment[s].k_len);
    causal_shift = kv_tokens - q_tokens;
  }
  // Queries of one unit head; unit head and its query block.
  const bool pack = QB == 1 && p.pack;
  const int rows = pack ? q_tokens * p.group : q_tokens;
  const int q_blocks = (rows + BLOCK_M - 1) / BLOCK_M;
  const int head_slot = slot / q_blocks;
  const int unit = head_slot + (p.numbering == kHeadsPerXcd ? (b & 7) * (p.unit_heads >> 3) : 0);
  const int in_head = slot - head_slot * q_blocks;
  const int q_block = (p.causal ? q_blocks - 1 - in_head : in_head) * BLOCK_M;

  const int tid = threadIdx.x;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int lane = tid & 63;
  const int r16 = lane & 15;  // query within a 16-query block; key / d row within a 16-row fragment
  const int j = lane >> 4;    // k-slot group
  const int kv_head = pack ? unit : unit / p.group;
  const int qw0 = q_block + wave * 16 * QB;

  // Row qw0 + 16 qb + r16 is query qi[qb] of query head `head` (with pack
  // that of this lane's row).
  const auto query_of = [&](int row) { return pack ? (int)((uint32_t)row / (uint32_t)p.group) : row; };
  int qi[QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) qi[qb] = query_of(qw0 + 16 * qb + r16);
  const int head = pack ? unit * p.group + (qw0 + r16 - qi[0] * p.group) : unit;

  const uint16_t* qp = p.q + (int64_t)q0 * p.sq_t + (int64_t)head * p.sq_h;
  const uint16_t* kp = p.k + (int64_t)k0 * p.sk_t + (int64_t)kv_head * p.sk_h;
  const uint16_t* vp = p.v + (int64_t)k0 * p.sv_t + (int64_t)kv_head * p.sv_h;

  // The last key query i sees is causal_base + i (and no key past the chunk).
  const int causal_base = p.q_local_offset + causal_shift - p.kv_local_offset;
  // Keys at or beyond kv_end are invisible to every query of this workgroup
  // and at or beyond wave_end to every query of this wave (a wave without
  // queries sees none); those before wave_first are visible to all of them.
  int kv_end = kv_tokens;
  int wave_end = qw0 < rows ? kv_tokens : 0;
  int wave_first = kv_tokens;
  if (p.causal) {
    kv_end = max(0, min(kv_end, causal_base + query_of(min(rows, q_block + BLOCK_M) - 1) + 1));
    wave_end = min(wave_end, causal_base + query_of(min(rows, qw0 + 16 * QB) - 1) + 1);
    wave_first = min(wave_first, causal_base + query_of(qw0) + 1);
  }
  const int ntiles = (kv_end + kTileKeys - 1) / kTileKeys;
  // The scale is fused into the exponent's FMA and the max is taken on raw
  // logits, which needs a positive factor: a negative scale was folded into
  // the sign of Q when the fragments were loaded, and a zero scale becomes
  // 1e-30 (every logit then rounds to the same exponent, as with zero).
  const float cf = scale_factor(p.scale_log2);

  // HBM/L2 -> LDS DMA of key tile [kt, kt + 64), issued by waves 0-3 (the
  // first wave of each SIMD) only.  The second waves of the SIMDs get the
  // smaller share of issue slots while both compute, so they finish a tile
  // last; the first waves wait at the tile barrier meanwhile, and issuing
  // the DMA there takes it off the tile's critical path.
  // Piece f of a tensor is LDS bytes [f KB, f KB + 1 KB), and each lane
  // loads the global granule the layouts above place at its slot.  The global
  // element offset is a wave-uniform part (f) plus a per-lane part (lane):
  //   K (fragment CK kb + c = f): key 16 (f / CK) + lane / 4, d 32 (f % CK)
  //   + 8 k_granule((lane % 4) ^ (lane / 16));
  //   V: key 16 (f % 4) + lane / 4, d 32 (f / 4) + 8 ((lane % 4) ^ 2 (lane / 16 % 2));
  //   V^T: the tile's bytes in order.
  // In the tail tile, keys past the chunk read its last key; granules past
  // head_dim read d = 0.  Those values are finite and masked (keys) or
  // multiplied by zero Q / never stored (d), and every address stays inside
  // the caller's buffers.
  // Wave-uniform byte address plus a 32-bit byte offset per lane: no vector
  // address arithmetic outside the edge tiles.
  auto dma = [](const uint16_t* base, uint32_t offset, uint8_t* dst) __attribute__((always_inline)) {
    asm volatile("" : "+s"(base));  // keeps the sum below uniform base + lane offset
    __builtin_amdgcn_global_load_lds((const SA_GLOBAL void*)(reinterpret_cast<const uint8_t*>(base) + offset),
                                     (SA_LDS void*)dst, 16, 0, 0);
  };
  auto issue_pieces = [&](int kt, uint8_t* stage, auto edge) __attribute__((always_inline)) {
    // Where registers are short the lane offsets are worked out anew for each
    // tile: held over the tile loop they cost head_dim 256 spills inside it
    // (4.7 us per tile instead of 3.5).
    int dma_lane = lane;
    if constexpr (QB > 1 && DP >= 128) asm volatile("" : "+v"(dma_lane));
    const int k_dma_d = 8 * Geo::k_granule((dma_lane & 3) ^ (dma_lane >> 4));
    const int v_dma_d = 8 * ((dma_lane & 3) ^ (2 * ((dma_lane >> 4) & 1)));
    const uint32_t k_dma_lane = 2u * ((dma_lane >> 2) * (uint32_t)p.sk_t + k_dma_d);
    const uint32_t v_dma_lane = VT ? 16u * dma_lane : 2u * ((dma_lane >> 2) * (uint32_t)p.sv_t + v_dma_d);
    uint8_t* k_stage = stage;
    uint8_t* v_stage = stage + Geo::TILE_BYTES;
    const uint16_t* kt_base = kp + (int64_t)kt * p.sk_t;
    const uint16_t* vt_base = VT ? vp + (int64_t)kt * DP : vp + (int64_t)kt * p.sv_t;
    const int last = kv_tokens - 1 - kt;  // last row of the chunk, in tile rows
#pragma unroll
    for (int i = 0; i < Geo::PIECES / Geo::ISSUERS; ++i) {
      const int f = wave * (Geo::PIECES / Geo::ISSUERS) + i;
      const int k_key0 = 16 * (f / CK);
      const int k_d0 = 32 * (f % CK);
      if constexpr (edge.value) {
        const int d = k_d0 + k_dma_d;
        const uint32_t row = min(k_key0 + (dma_lane >> 2), last);
        dma(kt_base, 2u * (row * (uint32_t)p.sk_t + (d < p.head_dim ? d : 0)), k_stage + f * 1024);
      } else {
        dma(kt_base + (int64_t)k_key0 * p.sk_t + k_d0, k_dma_lane, k_stage + f * 1024);
      }
      if constexpr (VT) {
        dma(vt_base + f * 512, v_dma_lane, v_stage + f * 1024);
      } else {
        const int v_key0 = 16 * (f & 3);
        const int v_d0 = 32 * (f >> 2);
        if constexpr (edge.value) {
          const int d = v_d0 + v_dma_d;
          const uint32_t row = min(v_key0 + (dma_lane >> 2), last);
          dma(vt_base, 2u * (row * (uint32_t)p.sv_t + (d < p.head_dim ? d : 0)), v_stage + f * 1024);
        } else {
          dma(vt_base + (int64_t)v_key0 * p.sv_t + v_d0, v_dma_lane, v_stage + f * 1024);
        }
      }
    }
  };
  auto issue_tile = [&](int kt, uint8_t* stage) __attribute__((always_inline)) {
    if (wave >= Geo::ISSUERS) return;
    if (kt + kTileKeys > kv_tokens || p.head_dim < DP)
      issue_pieces(kt, stage, std::true_type());
    else
      issue_pieces(kt, stage, std::false_type());
    __builtin_amdgcn_sched_barrier(0);
  };

  // The first tile's DMA is issued before the Q and state loads, so that it
  // is in flight while they arrive (the 16-bit path; the INT8 path stages
  // its own first tile).
  if constexpr (!QUANT) {
    if (ntiles > 0) issue_tile(0, lds_a);
  }

  // Q fragments: query qw0 + 16 qb + r16, d = 32 c + 8 j .. +7.  Rows and
  // granules past the end read the last query's d = 0 and are zeroed: loads
  // under a branch each waited for the one before.
  u32x4 qf[QB][CK];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const uint16_t* row = qp + (int64_t)min(qi[qb], q_tokens - 1) * p.sq_t;
#pragma unroll
    for (int c = 0; c < CK; ++c) {
      const int d = 32 * c + 8 * j;
      qf[qb][c] = *reinterpret_cast<const u32x4*>(row + (d < p.head_dim ? d : 0));
    }
  }
#pragma unroll
  for (int qb = 0; qb < QB; ++qb)
#pragma unroll
    for (int c = 0; c < CK; ++c)
      qf[qb][c] = qi[qb] < q_tokens && 32 * c + 8 * j < p.head_dim ? qf[qb][c] ^ q_sign(p.scale_log2) : u32x4{0, 0, 0, 0};

  // The ring's other tiles, behind the wait for Q.
  if constexpr (RING) {
    for (int t = 1; t < min(ntiles, STAGES - 1); ++t) issue_tile(t * kTileKeys, lds_a + t * STAGE_BYTES);
  }

  // Online-softmax state (base-2 domain); acc[db][qb] holds d = 16 db + 4 j
  // .. +3 of query qi[qb], l_part this lane's share of l.
  float m_run[QB], l_part[QB];
  f32x4 acc[DB][QB];
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    m_run[qb] = -INFINITY;
    l_part[qb] = 0.f;
#pragma unroll
    for (int db = 0; db < DB; ++db) acc[db][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
    if (!p.init && qi[qb] < q_tokens) {
      const int64_t blk = state_block(qi[qb], head, p.q_heads);
      const int r = qi[qb] & 15;  // r16, unless packed
      const int64_t srow = p.tiled_state ? blk * 16 + r : (int64_t)qi[qb] * p.ss_t + (int64_t)head * p.ss_h;
      m_run[qb] = p.m[srow];
      l_part[qb] = j == 0 ? p.l[srow] : 0.f;
      const float* arow = p.tiled_state ? p.acc + blk * 16 * p.head_dim + 4 * (16 * j + r)
                                        : p.acc + (int64_t)qi[qb] * p.sa_t + (int64_t)head * p.sa_h + 4 * j;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        if (16 * db + 4 * j < p.head_dim)
          acc[db][qb] = *reinterpret_cast<const f32x4*>(arow + (p.tiled_state ? 256 * db : 16 * db));
      }
    }
  }

  // Per-lane parts of the fragment addresses: 16 bytes per lane for the K and
  // V^T fragments, 8 bytes per lane for the transposing V reads (of an even d
  // block; an odd one's is at the other 32 bytes).
  const int k_lane = 64 * r16 + ((Geo::k_slot(j) ^ (r16 >> 2)) << 4);
  const int v_lane = VT ? 16 * lane : 256 * j + 64 * (r16 >> 2) + 32 * (j & 1) + 8 * (r16 & 3);
  const int v_lane_odd = v_lane ^ 32;

  // The MFMA / softmax work of tile t, read from the 16-bit stage `cur`.
  auto compute = [&](int t, const uint8_t* cur) {
    const int kt = t * kTileKeys;
    const uint8_t* k_stage = cur;
    const uint8_t* v_stage = cur + Geo::TILE_BYTES;
#pragma unroll
    for (int sub = 0; sub < kTileKeys / kSubKeys; ++sub) {
      const int rb = sub * kSubKeys;
      const int key0 = kt + rb;
      if (key0 >= wave_end) break;

      // S^T: two 16-key blocks x QB 16-query blocks, CK 32-wide d steps.
      f32x4 s[2][QB];
#pragma unroll
      for (int kb = 0; kb < 2; ++kb)
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) s[kb][qb] = f32x4{0.f, 0.f, 0.f, 0.f};
      const uint32_t k_addr = (uint32_t)(uintptr_t)(const SA_LDS uint8_t*)(k_stage) + k_lane;
#pragma unroll
      for (int c0 = 0; c0 < CK; c0 += KB) {
        // kf[kb KB + c]: 16-key block kb of the step, d step c0 + c.
        u32x4 kf[2 * KB];
        read_k(kf, k_addr, (rb / 16 * CK + c0) * 1024, CK * 1024);
        // Query blocks in snake order: consecutive MFMAs change only one of
        // their A and B operands except where c changes.  An MFMA whose A
        // and B both differ from the previous one's issues later (measured:
        // up to 1.5x the MFMA's cycles).
#pragma unroll
        for (int c = 0; c < KB; ++c)
#pragma unroll
          for (int kb = 0; kb < 2; ++kb)
#pragma unroll
            for (int i = 0; i < QB; ++i) {
              const int qb = kb == 0 ? i : QB - 1 - i;
              s[kb][qb] = Op::mma(kf[kb * KB + c], qf[qb][c0 + c], s[kb][qb]);
            }
      }

      if (__builtin_expect(key0 + kSubKeys > wave_first, 0)) {
#pragma unroll
        for (int kb = 0; kb < 2; ++kb)
#pragma unroll
          for (int qb = 0; qb < QB; ++qb)
#pragma unroll
            for (int i = 0; i < 4; ++i) {
              const int key = key0 + 16 * kb + 4 * j + i;
              const bool ok = key < kv_tokens && (!p.causal || key <= causal_base + qi[qb]);
              s[kb][qb][i] = ok ? s[kb][qb][i] : -INFINITY;
            }
      }

      // P^T against the kept maximum, and the lane's partial row sum (8 keys).
      // The pairwise sum order is fixed, so a row's sum does not depend on
      // which path computed it.
      auto exps = [&](int qb, float neg_m, u32x4& pq) -> float {
        float sum = 0.f;
#pragma unroll
        for (int kb = 0; kb < 2; ++kb) {
#pragma unroll
          for (int e = 0; e < 2; ++e) {
            const float p0 = __builtin_amdgcn_exp2f(fmaf(s[kb][qb][2 * e], cf, neg_m));
            const float p1 = __builtin_amdgcn_exp2f(fmaf(s[kb][qb][2 * e + 1], cf, neg_m));
            sum = (kb == 0 && e == 0) ? p0 + p1 : sum + (p0 + p1);
            pq[2 * kb + e] = Op::pack2(p0, p1);
          }
        }
        return sum;
      };
      u32x4 pf[QB];
      float psum[QB];
      bool grow[QB];
      bool any = false;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        // Every p <= 2^8 (no logit above m + 8) whenever the lane's sum is.
        // Against m = -inf (no maximum yet) every p is inf, or NaN where the
        // key is masked, so such a row always takes the rescale path.
        psum[qb] = exps(qb, -m_run[qb], pf[qb]);
        grow[qb] = !(psum[qb] <= 256.f);
        any = any || grow[qb];
      }
      // Rescale only when some logit of the wave may have left the [.., m + 8]
      // window; where m stays, the values computed above stand.
      if (__builtin_expect(__ballot(any) != 0, 0)) {
#pragma unroll
        for (int qb = 0; qb < QB; ++qb) {
          // The query's own decision: one of its four lanes saw a partial sum
          // above 2^8 (some logit may exceed m + 8) or it has no maximum yet.
          const uint64_t bal = __ballot(grow[qb]);
          uint32_t fold = (uint32_t)bal | (uint32_t)(bal >> 32);
          fold |= fold >> 16;
          const bool mine = (fold >> r16) & 1u;
          float a = fmaxf(fmaxf(s[0][qb][0], s[0][qb][1]), fmaxf(s[0][qb][2], s[0][qb][3]));
          a = fmaxf(a, fmaxf(fmaxf(s[1][qb][0], s[1][qb][1]), fmaxf(s[1][qb][2], s[1][qb][3]))) * cf;
          float full = fmaxf(a, __shfl_xor(a, 16));
          full = fmaxf(full, __shfl_xor(full, 32));
          const float m_new = (mine && full > m_run[qb] + kRescaleThreshold) ? full : m_run[qb];
          // Without a maximum yet masked keys weigh 0 and NaN stays NaN.
          const bool none = m_new == -INFINITY;
          if (m_new != m_run[qb] || none) {
            const float alpha = none ? 1.f : __builtin_amdgcn_exp2f(m_run[qb] - m_new);
            l_part[qb] *= alpha;
#pragma unroll
            for (int db = 0; db < DB; ++db) acc[db][qb] *= alpha;
            m_run[qb] = m_new;
            psum[qb] = exps(qb, none ? 0.f : -m_new, pf[qb]);
          }
        }
      }
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) l_part[qb] += psum[qb];

      // O^T += V^T P^T, VB d blocks per batch of LDS reads.
      const uint32_t v_base = (uint32_t)(uintptr_t)(const SA_LDS uint8_t*)(v_stage);
      const uint32_t v_addr = v_base + v_lane;
      const uint32_t v_addr_odd = v_base + v_lane_odd;
#pragma unroll
      for (int d0 = 0; d0 < DB; d0 += VB) {
        // Rows d = 16 db + r16 of V^T, key granule j of the step's 32-key
        // block.  From V's rows lane (j, r16) addresses key 4 j + r16 / 4 of
        // each 16-key block at d = 16 db + 4 (r16 % 4) .. +3; after the
        // transpose it holds d = 16 db + r16 for keys 4 j .. 4 j + 3.
        u32x4 vf[VB];
        if constexpr (VT)
          read_vt(vf, v_addr, (rb / 32 * DB + d0) * 1024);
        else
          read_v(vf, v_addr, v_addr_odd, d0 / 2 * 4096 + rb * 64);
#pragma unroll
        for (int dd = 0; dd < VB; ++dd)
#pragma unroll
          for (int i = 0; i < QB; ++i) {
            const int qb = dd % 2 == 0 ? i : QB - 1 - i;  // snake order, as in QK^T
            acc[d0 + dd][qb] = Op::mma(vf[dd], pf[qb], acc[d0 + dd][qb]);
          }
      }
    }
  };

  // Sum of a query's four partial row sums, identical on all four lanes.
  auto full_l = [&](float x) -> float {
    const float h = x + __shfl_xor(x, 16);
    return h + __shfl_xor(h, 32);
  };

  int until_merge = p.merge_tiles;  // tiles left in the current K/V chunk
  auto merge_after_tile = [&]() {
    if (p.merge_tiles > 0 && --until_merge == 0) {
      until_merge = p.merge_tiles;
#pragma unroll
      for (int qb = 0; qb < QB; ++qb) {
        const float full = full_l(l_part[qb]);
        l_part[qb] = j == 0 ? full : 0.f;
      }
    }
  };
  if constexpr (RING) {
    // As below, with tiles t+1 .. t+STAGES-2 in flight across the barrier.
    // An issuing wave's DMA completes in order, PER_TILE of them per tile, so
    // tile t is there once no more than the later tiles' are outstanding.
    constexpr int PER_TILE = 2 * Geo::PIECES / Geo::ISSUERS;
    static_assert((STAGES - 2) * PER_TILE <= 63, "vmcnt range");
    for (int t = 0; t < ntiles; ++t) {
      const int later = ntiles - 1 - t;
      if (later >= 2)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(2 * PER_TILE) : "memory");
      else if (later == 1)
        asm volatile("s_waitcnt vmcnt(%0)" ::"n"(PER_TILE) : "memory");
      else
        asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (later >= STAGES - 1)
        issue_tile((t + STAGES - 1) * kTileKeys, lds_a + ((t + STAGES - 1) & (STAGES - 1)) * STAGE_BYTES);
      compute(t, lds_a + (t & (STAGES - 1)) * STAGE_BYTES);
      merge_after_tile();
    }
  } else if constexpr (!QUANT) {
    // Tile t is computed from `cur` while tile t+1 streams into `next`.
    auto tile = [&](int t, const uint8_t* cur, uint8_t* next) {
      // Every wave waits for its own DMA of tile t before the barrier, so
      // after it all 64 rows of `cur` are in LDS.  LDS DMA is counted by
      // vmcnt, which a workgroup-scope fence does not wait for: without this
      // explicit wait a wave could read rows that another wave's DMA has not
      // written yet.  The barrier also guarantees `next` (tile t-1) is no
      // longer being read.
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (t + 1 < ntiles) issue_tile((t + 1) * kTileKeys, next);
      compute(t, cur);
      merge_after_tile();
    };
    for (int t = 0; t < ntiles; t += 2) {
      tile(t, lds_a, lds_b);
      if (t + 1 < ntiles) tile(t + 1, lds_b, lds_a);
    }
  } else {
    // Raw int8 tile [kt, kt + 64) of K and V into staging `stg` (K at 0, V at
    // I8_TILE_BYTES), row-major with 16-byte granules; wave w moves KB w of
    // each.  The same tail and head_dim clamps as the 16-bit path keep every
    // address in the buffers.
    const uint8_t* kp8 = reinterpret_cast<const uint8_t*>(p.k) + (int64_t)kv_head * p.sk_h;
    const uint8_t* vp8 = reinterpret_cast<const uint8_t*>(p.v) + (int64_t)kv_head * p.sv_h;
    const int row8 = wave * (1024 / DP) + lane / Geo::I8_GR;
    const int col8 = (lane % Geo::I8_GR) * 16 < p.head_dim ? (lane % Geo::I8_GR) * 16 : 0;
    auto issue_i8 = [&](int kt, uint8_t* stg) {
      if (wave >= Geo::I8_DMAS) return;
      const int row = min(kt + row8, kv_tokens - 1);
      __builtin_amdgcn_global_load_lds((const SA_GLOBAL void*)(kp8 + (int64_t)row * p.sk_t + col8),
                                       (SA_LDS void*)(stg + wave * 1024), 16, 0, 0);
      __builtin_amdgcn_global_load_lds((const SA_GLOBAL void*)(vp8 + (int64_t)row * p.sv_t + col8),
                                       (SA_LDS void*)(stg + Geo::I8_TILE_BYTES + wave * 1024), 16, 0, 0);
    };
    // This thread's dequantization granule: row tid / I8_GR of the tile.  Its
    // scales (raw fp16 bits) are loaded one tile ahead into registers.
    uint32_t ksc = 0, vsc = 0;
    const uint16_t* ksp = p.ks + (int64_t)kv_head * p.sks_h;
    const uint16_t* vsp = p.vs + (int64_t)kv_head * p.svs_h;
    const bool dequantizes = tid < Geo::I8_GRANULES;
    auto load_scales = [&](int kt) {
      if (!dequantizes) return;
      const int key = min(kt + tid / Geo::I8_GR, kv_tokens - 1);
      const int64_t group = (int64_t)((p.scale_offset + key) >> p.scale_shift);
      ksc = ksp[group * p.sks_g];
      vsc = vsp[group * p.svs_g];
    };
    // dtype(fp32(k) * fp32(scale)) into the 16-bit stage.  A signed byte b is
    // (b ^ 0x80) - 128; fma(u, s, -128 s) rounds (u - 128) * s once, the same
    // value as the reference's fp32 product.
    auto dequant = [&](const uint8_t* stg, uint8_t* stage) {
      if (!dequantizes) return;
      const int row = tid / Geo::I8_GR;
      const int gr = tid % Geo::I8_GR;
#pragma unroll
      for (int tensor = 0; tensor < 2; ++tensor) {
        const u32x4 raw = *reinterpret_cast<const u32x4*>(stg + tensor * Geo::I8_TILE_BYTES + row * DP + gr * 16);
        const uint16_t bits = (uint16_t)(tensor == 0 ? ksc : vsc);
        const float sc = (float)__builtin_bit_cast(_Float16, bits);
        const float nb = -128.f * sc;
        u32x4 out[2];
#pragma unroll
        for (int w = 0; w < 4; ++w) {
          const uint32_t x = raw[w] ^ 0x80808080u;
          const float f0 = fmaf((float)(x & 0xffu), sc, nb);
          const float f1 = fmaf((float)((x >> 8) & 0xffu), sc, nb);
          const float f2 = fmaf((float)((x >> 16) & 0xffu), sc, nb);
          const float f3 = fmaf((float)(x >> 24), sc, nb);
          out[w >> 1][2 * (w & 1)] = Op::pack2(f0, f1);
          out[w >> 1][2 * (w & 1) + 1] = Op::pack2(f2, f3);
        }
        if (tensor == 0) {
          *reinterpret_cast<u32x4*>(stage + Geo::k_offset(row, 2 * gr)) = out[0];
          *reinterpret_cast<u32x4*>(stage + Geo::k_offset(row, 2 * gr + 1)) = out[1];
        } else {
          *reinterpret_cast<u32x4*>(stage + Geo::TILE_BYTES + Geo::v_offset(row, 2 * gr)) = out[0];
          *reinterpret_cast<u32x4*>(stage + Geo::TILE_BYTES + Geo::v_offset(row, 2 * gr + 1)) = out[1];
        }
      }
    };
    // At tile t: `cur` holds tile t (dequantized before the barrier), staging
    // `stg_next` holds raw tile t+1 and `stg_cur` (raw tile t) and `next`
    // (read by tile t-1's MFMAs) are free.  The vmcnt wait covers this wave's
    // DMA and scale loads; the barrier makes every wave's DMA and
    // dequantization writes visible.
    auto tile_q = [&](int t, const uint8_t* cur, uint8_t* next, uint8_t* stg_cur, const uint8_t* stg_next) {
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      if (t + 2 < ntiles) issue_i8((t + 2) * kTileKeys, stg_cur);
      // The first wave of a SIMD dequantizes before its MFMAs and the second
      // one after them, so that each wave's vector work meets the other's
      // matrix work (head_dim 128, 16 / 32 / 48 queries per wave: 1.91 / 2.65
      // / 3.27 us per tile with all waves first, 1.73 / 2.50 / 3.20 so).
      auto dequant_next = [&]() {
        if (t + 1 < ntiles) {
          dequant(stg_next, next);
          if (t + 2 < ntiles) load_scales((t + 2) * kTileKeys);
        }
      };
      if (wave < Geo::ISSUERS) dequant_next();
      compute(t, cur);
      if (wave >= Geo::ISSUERS) dequant_next();
    };
    if (ntiles > 0) {
      issue_i8(0, lds_qa);
      load_scales(0);
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();
      dequant(lds_qa, lds_a);
      if (ntiles > 1) {
        issue_i8(kTileKeys, lds_qb);
        load_scales(kTileKeys);
      }
    }
    for (int t = 0; t < ntiles; t += 2) {
      tile_q(t, lds_a, lds_b, lds_qa, lds_qb);
      if (t + 1 < ntiles) tile_q(t + 1, lds_b, lds_a, lds_qb, lds_qa);
    }
  }

  // The epilogue's parameters are read from the kernel's argument memory
  // again: kept in scalar registers across the tile loop they displaced its
  // own (the scalar spills took vector registers).
  asm volatile("" : "+s"(args));
  const SA_CONSTANT UpdateParams& e = *args;
#pragma unroll
  for (int qb = 0; qb < QB; ++qb) {
    const float l_full = full_l(l_part[qb]);
    if (qi[qb] >= q_tokens) continue;
    if (e.out != nullptr) {
      uint16_t* orow = e.out + (int64_t)(q0 + qi[qb]) * e.so_t + (int64_t)head * e.so_h + 4 * j;
#pragma unroll
      for (int db = 0; db < DB; ++db) {
        if (16 * db + 4 * j < e.head_dim) {
          const f32x4& a = acc[db][qb];
          u32x2 o = {0, 0};
          if (l_full > 0.f) {
            o[0] = Op::pack2(a[0] / l_full, a[1] / l_full);
            o[1] = Op::pack2(a[2] / l_full, a[3] / l_full);
          }
          *reinterpret_cast<u32x2*>(orow + 16 * db) = o;
        }
      }
      if (e.lse != nullptr && j == 0)
        e.lse[(int64_t)head * e.lse_sh + e.lse_off + q0 + qi[qb]] =
            l_full > 0.f ? (m_run[qb] + log2f(l_full)) * 0.69314718055994530942f : -INFINITY;
      continue;
    }
    const int64_t blk = state_block(qi[qb], head, e.q_heads);
    const int r = qi[qb] & 15;
    const int64_t srow = e.tiled_state ? blk * 16 + r : (int64_t)qi[qb] * e.ss_t + (int64_t)head * e.ss_h;
    if (j == 0) {
      e.m[srow] = m_run[qb];
      e.l[srow] = l_full;
    }
    float* arow = e.tiled_state ? e.acc + blk * 16 * e.head_dim + 4 * (16 * j + r)
                                : e.acc + (int64_t)qi[qb] * e.sa_t + (int64_t)head * e.sa_h + 4 * j;
#pragma unroll
    for (int db = 0; db < DB; ++db) {
      if (16 * db + 4 * j < e.head_dim)
        *reinterpret_cast<f32x4*>(arow + (e.tiled_state ? 256 * db : 16 * db)) = acc[db][qb];
    }
  }
}

template <typename Op, int DP, int QB, int MODE>
hipError_t launch_kernel(const UpdateParams& p, const LaunchShape& shape, hipStream_t stream) {
  if constexpr (QB == 1 && MODE == kRows && DP <= 128) {
    if (shape.stages == 4) {
      hipLaunchKernelGGL((update_kernel<Op, DP, QB, MODE, 4>), dim3(shape.grid), dim3(Geometry<DP>::THREADS), 0, stream, p);
      return hipGetLastError();
    }
  }
  hipLaunchKernelGGL((update_kernel<Op, DP, QB, MODE, 2>), dim3(shape.grid), dim3(Geometry<DP>::THREADS), 0, stream, p);
  return hipGetLastError();
}

template <int DP, int QB, int MODE>
hipError_t launch_variant(const UpdateParams& p, const LaunchShape& shape, int dtype, hipStream_t stream) {
  static_assert(Geometry<DP>::THREADS == kThreads && Geometry<DP>::WAVES * 16 == kRowsPerBlock, "launch shape");
  return dtype == SA_DTYPE_BF16 ? launch_kernel<BF16, DP, QB, MODE>(p, shape, stream)
                                : launch_kernel<FP16, DP, QB, MODE>(p, shape, stream);
}

}  // namespace
}  // namespace sa
