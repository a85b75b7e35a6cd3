// Launchers of the chunk-update kernel (sa_update_kernel.h), and the finalize
// and V-transpose kernels of the streamed exact-attention path for MI355X
// (gfx950, CDNA4).
//
// The finalize kernel follows _finalize_attention_kernel (reference
// src/seqattn_core/kernels/streaming.py:158-202): out = acc / l (0 where
// l == 0); it also writes LSE = (m + log2 l) * ln 2, which the reference does
// not produce.

#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstdint>
#include <mutex>
#include <new>
#include <vector>

#include "sa_common.h"
#include "sa_update_kernel.h"

namespace sa {
namespace {

struct FinalizeParams {
  const float* acc;
  const float* m;
  const float* l;
  uint16_t* out;
  float* lse;
  int64_t sa_t, sa_h, ss_t, ss_h, so_t, so_h, lse_sh, lse_off;
  int32_t q_tokens, q_heads, groups;  // groups = head_dim / 8
  int32_t tiled_state;  // state in the row-group layout (state_block)
};

// One workgroup per (16-row group, head): blockIdx.x is the row group and
// blockIdx.y the head, so no thread divides 64-bit indices.  Item i of the
// group covers row r = i % 16 and output granule g = i / 16 (d = 8g .. 8g +
// 7).  In the row-group layout a wave's 64 items read 2 KB of consecutive
// accumulator bytes (chunks 2g and 2g + 1 of 16 rows) and write 16 rows x 64
// bytes of output.
template <typename Op>
__global__ __launch_bounds__(256) void finalize_kernel(const FinalizeParams p) {
  const int h = blockIdx.y;
  const int64_t row0 = (int64_t)blockIdx.x * 16;
  const int64_t blk = state_block(row0, h, p.q_heads);
  const int items = 16 * p.groups;
  for (int i = threadIdx.x; i < items; i += 256) {
    const int r = i & 15;
    const int g = i >> 4;
    const int64_t t = row0 + r;
    if (t >= p.q_tokens) continue;
    const int64_t srow = p.tiled_state ? blk * 16 + r : t * p.ss_t + h * p.ss_h;
    const float l = p.l[srow];
    f32x4 a0, a1;
    if (p.tiled_state) {
      // Chunks 2g and 2g + 1 (d = 8g .. 8g + 7) of row r.
      const float* a = p.acc + blk * 16 * (p.groups * 8) + (2 * g * 16 + r) * 4;
      a0 = *reinterpret_cast<const f32x4*>(a);
      a1 = *reinterpret_cast<const f32x4*>(a + 16 * 4);
    } else {
      const float* a = p.acc + t * p.sa_t + h * p.sa_h + 8 * g;
      a0 = *reinterpret_cast<const f32x4*>(a);
      a1 = *reinterpret_cast<const f32x4*>(a + 4);
    }
    u32x4 o;
    if (l > 0.f) {
      o[0] = Op::pack2(a0[0] / l, a0[1] / l);
      o[1] = Op::pack2(a0[2] / l, a0[3] / l);
      o[2] = Op::pack2(a1[0] / l, a1[1] / l);
      o[3] = Op::pack2(a1[2] / l, a1[3] / l);
    } else {
      o = u32x4{0, 0, 0, 0};
    }
    *reinterpret_cast<u32x4*>(p.out + t * p.so_t + h * p.so_h + 8 * g) = o;
    if (p.lse != nullptr && g == 0) {
      const float m = p.m[srow];
      p.lse[h * p.lse_sh + p.lse_off + t] = l > 0.f ? (m + log2f(l)) * 0.69314718055994530942f : -INFINITY;
    }
  }
}

// Transposed copy of V for the head_dim-128 update kernel's kTransposedV mode.
// V is [kv_tokens, kv_heads, 128] with element strides (sv_t, sv_h); vt is
// [kv_heads][t_pad / 64] tiles of 64 keys x 128 d, each in the order of the
// kernel's LDS stage, so that the kernel's tile DMA reads consecutive bytes:
// 16-byte piece i of a tile is fragment i / 64 (32-key group i / 512, d block
// i / 64 % 8), lane i % 64: row d = 16 (i / 64 % 8) + i % 16, slots 8 j ..
// 8 j + 7 with j = i / 16 % 4, which hold keys 4j .. 4j + 3 and 16 + 4j ..
// 16 + 4j + 3 of the group, the k-slot order in which that kernel's P^T
// operand holds the keys of a 16x16x32 MFMA.  Keys kv_tokens .. t_pad-1 are
// zero.  One workgroup per (kv_head, 64 keys), staged through LDS.
struct TransposeParams {
  const uint16_t* v;
  uint16_t* vt;
  int64_t sv_t, sv_h, t_pad;
  int32_t kv_tokens, tiles;
};

__global__ __launch_bounds__(256) void transpose_v_kernel(const TransposeParams p) {
  __shared__ __attribute__((aligned(16))) uint16_t tile[64][128 + 8];
  const int tid = threadIdx.x;
  const int head = blockIdx.x / p.tiles;
  const int kt = (blockIdx.x - head * p.tiles) * 64;
  {
    // Thread t reads key kt + t / 4, elements 32 (t % 4) .. +31.
    const int key = tid >> 2, d0 = (tid & 3) * 32;
    const bool ok = kt + key < p.kv_tokens;
    const uint16_t* src = p.v + (int64_t)(kt + key) * p.sv_t + (int64_t)head * p.sv_h + d0;
#pragma unroll
    for (int j = 0; j < 4; ++j) {
      const u32x4 w = ok ? *reinterpret_cast<const u32x4*>(src + 8 * j) : u32x4{0, 0, 0, 0};
      *reinterpret_cast<u32x4*>(&tile[key][d0 + 8 * j]) = w;
    }
  }
  __syncthreads();
  {
    uint16_t* dst = p.vt + (int64_t)head * 128 * p.t_pad + (int64_t)kt * 128;
#pragma unroll
    for (int n = 0; n < 4; ++n) {
      const int i = n * 256 + tid;
      const int d = 16 * ((i >> 6) & 7) + (i & 15);
      const int key = 32 * (i >> 9) + 4 * ((i >> 4) & 3);
      u32x4 w;
#pragma unroll
      for (int e = 0; e < 4; ++e) {
        const int k = key + 16 * (e >> 1) + 2 * (e & 1);
        w[e] = (uint32_t)tile[k][d] | ((uint32_t)tile[k + 1][d] << 16);
      }
      *reinterpret_cast<u32x4*>(dst + 8 * i) = w;
    }
  }
}

constexpr int kCUs = 256;

int64_t tiles_of(int64_t keys) { return (std::max<int64_t>(0, keys) + kTileKeys - 1) / kTileKeys; }

// Modelled time (in the units of kVariants) of the launch with workgroups of
// v.rows queries, from the measured time per tile.  Blocks of equal length
// run in rounds of one (or two) workgroups per CU; under a causal mask and
// with several segments long blocks start first and short ones fill in behind
// them, and a launch that shares the chip with another one fills in behind
// that.  No launch ends before its longest block.  Over 60 drawn launches the
// chosen width took 0.8% more than the best one on average, 6.7% at most.
double variant_time(const UpdateVariant& v, const UpdateParams& p, bool overlapped) {
  // The narrowest workgroups pack the query heads of a K/V head.
  const int64_t group = v.rows == kVariants[0][0].rows ? p.group : 1;
  double longest = 0, shortest = 0, work = 0, n = 0;
  const auto add = [&](int64_t q_len, int64_t k_len, int64_t first_visible) {
    const double blocks = (double)((q_len * group + v.rows - 1) / v.rows) * (p.q_heads / group);
    // Tiles of the last and the first block.
    const double last = tiles_of(p.causal ? std::min(k_len, first_visible + q_len - 1) : k_len);
    const double first =
        p.causal ? tiles_of(std::min(k_len, first_visible + std::min<int64_t>(v.rows / group, q_len) - 1)) : last;
    longest = std::max(longest, last);
    shortest = n == 0 ? first : std::min(shortest, first);
    work += 0.5 * (first + last) * blocks;
    n += blocks;
  };
  if (p.segments > 1) {
    for (int s = 0; s < p.segments; ++s)
      add(p.segment[s].q_len, p.segment[s].k_len, p.segment[s].k_len - p.segment[s].q_len + 1);
  } else {
    add(p.q_tokens, p.kv_tokens, (int64_t)p.q_local_offset + p.causal_shift - p.kv_local_offset + 1);
  }
  if (n <= kCUs) return longest * v.one;
  const double slots = v.two ? 2 * kCUs : kCUs, slot = v.two ? v.two : v.one;
  const double even = work / slots * slot;
  if (overlapped) return std::max(longest * v.one, even);
  if (longest == shortest) {
    const double full = std::floor(n / slots), rest = n - full * slots;
    const double partly = rest == 0     ? 0.0
                          : rest <= kCUs ? v.one
                                         : v.one + (slot - v.one) * (rest - kCUs) / kCUs;
    return (full * slot + partly) * longest;
  }
  // Longest first: within one shortest block of an even spread, and no worse
  // than rounds of falling length.
  const double rounds = std::ceil(n / slots);
  const double in_rounds = rounds * slot * (longest - (longest - shortest) * 0.5 * (rounds - 1) * slots / n);
  return std::max(longest * v.one, std::min(in_rounds, even + shortest * slot));
}

// Queries per workgroup.  A query's bits do not depend on it, so it is chosen
// for time alone: wide workgroups read each K/V tile for more queries (bf16,
// head_dim 128: 6.1 ns per query and tile at 384 queries, 7.6 at 128), narrow
// ones fill the chip with few queries and waste less of a last round or of a
// causal diagonal.  1,009 queries over 61,312 keys x 32 heads: 384 queries
// are 96 workgroups, 128 are 256.
int choose_rows(const UpdateParams& p, int d, int mode, bool overlapped) {
  int rows = kVariants[d][0].rows;
  double best = -1.0;
  for (UpdateVariant v : kVariants[d]) {
    if (!v.rows) continue;
    if (mode == kInt8) {
      // Dequantizing a tile takes about 4 ns per padded d, and the staging of
      // head_dim 128 leaves LDS for one workgroup.
      v.one += 4 * (32 << d);
      v.two = d == 2 ? 0 : v.two + 8 * (32 << d);
    }
    const double t = variant_time(v, p, overlapped);
    // Ties go to the wider workgroup (less traffic).
    if (best < 0.0 || t <= best) best = t, rows = v.rows;
  }
  return rows;
}

// Numbers the launch's workgroups of `rows` rows (p's pack, unit_heads,
// numbering, first, slots and xcd_run) and returns how many there are.
uint32_t number_workgroups(UpdateParams& p, int rows) {
  const bool several = p.segments > 1;
  int64_t most_queries = several ? 0 : p.q_tokens;
  for (int s = 0; several && s < p.segments; ++s) most_queries = std::max<int64_t>(most_queries, p.segment[s].q_len);
  p.pack = rows == kRowsPerBlock && p.group > 1 && most_queries * p.group <= INT32_MAX;
  p.unit_heads = p.pack ? p.q_heads / p.group : p.q_heads;
  p.numbering = p.unit_heads % 8 == 0 ? kHeadsPerXcd : p.causal || several ? kDealt : kRunsPerXcd;
  const int heads = p.numbering == kHeadsPerXcd ? p.unit_heads / 8 : p.unit_heads;
  const int per_query = p.pack ? p.group : 1;
  p.slots = 0;
  for (int s = 0; s < (several ? p.segments : 1); ++s) {
    p.first[s] = p.slots;
    const int64_t queries = several ? p.segment[s].q_len : p.q_tokens;
    p.slots += (int32_t)((queries * per_query + rows - 1) / rows * heads);
  }
  p.xcd_run = (p.slots + 7) / 8;
  return p.numbering == kHeadsPerXcd ? 8u * p.slots : p.numbering == kDealt ? p.slots : 8u * p.xcd_run;
}

// LDS stages of a launch.  With two, a workgroup alone on its CU waits at
// every barrier for the tile it just requested; with four it has three tiles
// in flight, but starts later and runs a slightly longer loop.  Measured with
// both forced (head_dim 32 to 128, 1 to 24 segments, 1 to 256 queries, heads
// numbered in each of the three ways, which makes no difference):
//   K and V from HBM, time with four over two stages.  Rows for one wave: 0.99
//   to 1.05 at 256 keys, 0.91-1.0 at 512, 0.84-0.94 at 1,024, 0.71-0.91 from
//   4,096 (1.0 where 256 workgroups read heads of their own).  Rows for all
//   waves: 1.03-1.15 at 256, 1.0-1.1 at 512, 0.96-1.05 at 1,024, 0.90-1.04 at
//   2,048, 0.85-1.0 from 8,192.
//   K and V still in the 256 MB Infinity Cache from an earlier call: 0.99-1.06
//   at 1,024 keys, 1.02-1.09 above.
// So the line is where a program is likely to read them from HBM: over 32 MB
// a step through eight layers, or much else in between, has replaced them.
// Workgroups that share a CU hide each other's waits (head_dim 64, 420
// workgroups: 42.7 us with two stages, 43.5 with four).
int choose_stages(const UpdateParams& p, int d, int mode, int rows, uint32_t grid, bool overlapped) {
  if (mode != kRows || d > 2 || rows != kRowsPerBlock) return 2;
  int64_t keys = p.segments > 1 ? 0 : p.kv_tokens;
  for (int s = 0; p.segments > 1 && s < p.segments; ++s) keys += p.segment[s].k_len;
  const int64_t bytes = 4 * keys * (p.q_heads / p.group) * p.head_dim;
  const bool alone = grid <= (uint32_t)(overlapped ? kCUs / 2 : kCUs);
  int64_t most_queries = p.segments > 1 ? 0 : p.q_tokens;
  for (int s = 0; p.segments > 1 && s < p.segments; ++s) most_queries = std::max<int64_t>(most_queries, p.segment[s].q_len);
  const bool one_wave = most_queries * (p.pack ? p.group : 1) <= 16;
  const bool long_enough = keys >= int64_t(one_wave ? 512 : 1024) * std::max(1, p.segments);
  return alone && bytes > (int64_t(32) << 20) && long_enough ? 4 : 2;
}

int padded_head_dim(int head_dim) { return head_dim <= 32 ? 0 : head_dim <= 64 ? 1 : head_dim <= 128 ? 2 : 3; }

LaunchShape shape_launch(UpdateParams& p, int mode, bool overlapped) {
  const int d = padded_head_dim(p.head_dim);
  LaunchShape shape;
  shape.rows = choose_rows(p, d, mode, overlapped);
  shape.grid = number_workgroups(p, shape.rows);
  shape.stages = choose_stages(p, d, mode, shape.rows, shape.grid, overlapped);
  return shape;
}

// A launch has fewer than 2^32 threads (numbering rounds its workgroups up by
// at most 7).
constexpr int64_t kMaxWorkgroups = (int64_t(1) << 32) / kThreads - 8;

hipError_t launch_one(UpdateParams p, int mode, int dtype, bool overlapped, hipStream_t stream) {
  const LaunchShape shape = shape_launch(p, mode, overlapped);
  switch (padded_head_dim(p.head_dim)) {
    case 0: return launch_update_d32(p, mode, shape, dtype, stream);
    case 1: return launch_update_d64(p, mode, shape, dtype, stream);
    case 2: return launch_update_d128(p, mode, shape, dtype, stream);
    default: return launch_update_d256(p, mode, shape, dtype, stream);
  }
}

// More queries than one launch's workgroups hold go in several launches of
// consecutive rows (a query's bits do not depend on its neighbours).
hipError_t launch_update_variant(UpdateParams p, int mode, int dtype, bool overlapped, hipStream_t stream) {
  // A common multiple of the widths and of the state's 16-row groups.
  constexpr int64_t kStep = 768;
  const int64_t most = (kMaxWorkgroups / p.q_heads - 1) * kRowsPerBlock / kStep * kStep;
  while (p.segments <= 1 && most > 0 && p.q_tokens > most) {
    UpdateParams part = p;
    part.q_tokens = (int32_t)most;
    const hipError_t err = launch_one(part, mode, dtype, overlapped, stream);
    if (err != hipSuccess) return err;
    p.q += most * p.sq_t;
    p.q_local_offset += (int32_t)most;
    p.q_tokens -= (int32_t)most;
    if (p.out != nullptr) p.out += most * p.so_t;
    p.lse_off += most;
    if (p.m != nullptr) {
      p.m += most * (p.tiled_state ? p.q_heads : p.ss_t);
      p.l += most * (p.tiled_state ? p.q_heads : p.ss_t);
      p.acc += most * (p.tiled_state ? (int64_t)p.q_heads * p.head_dim : p.sa_t);
    }
  }
  return launch_one(p, mode, dtype, overlapped, stream);
}

// The segments of one call in launches of up to kMaxSegments, those with the
// most keys first: the workgroups of one launch run side by side, where a
// launch per segment left CUs idle at the end of each (11 ragged segments of
// 1,800 tokens x 32 heads on average: 11 launches of 38-86 us one after the
// other).
int32_t launch_segments(UpdateParams p, const FusedOutput& fused, int dtype, bool overlapped, hipStream_t stream) {
  std::vector<Segment> order;
  order.reserve(fused.num_segments);
  for (int32_t s = 0; s < fused.num_segments; ++s)
    if (fused.segments[s].q_len > 0) order.push_back(fused.segments[s]);
  std::stable_sort(order.begin(), order.end(), [](const Segment& a, const Segment& b) { return a.k_len > b.k_len; });
  for (size_t at = 0; at < order.size();) {
    int64_t workgroups = 0;
    p.segments = 0;
    while (at < order.size() && p.segments < kMaxSegments) {
      const int64_t more = ((int64_t)order[at].q_len + 127) / 128 * p.q_heads;
      if (p.segments > 0 && workgroups + more > kMaxWorkgroups) break;
      workgroups += more;
      p.segment[p.segments++] = order[at++];
    }
    UpdateParams one = p;
    if (p.segments == 1) {
      const Segment& seg = p.segment[0];
      one.q += (int64_t)seg.q0 * p.sq_t;
      one.k += (int64_t)seg.k0 * p.sk_t;
      one.v += (int64_t)seg.k0 * p.sv_t;
      one.out += (int64_t)seg.q0 * p.so_t;
      one.lse_off += seg.q0;
      one.q_tokens = seg.q_len;
      one.kv_tokens = seg.k_len;
      one.causal_shift = seg.k_len - seg.q_len;
    }
    const hipError_t err = launch_update_variant(one, kRows, dtype, overlapped, stream);
    if (err != hipSuccess) return hip_status(err, "update kernel launch");
  }
  return 0;
}

inline bool aligned(const void* ptr, uintptr_t n) { return (reinterpret_cast<uintptr_t>(ptr) % n) == 0; }

}  // namespace

int32_t update_block_rows(int32_t head_dim) {
  if (head_dim > 64 && head_dim <= 128) return 384;
  return head_dim <= 64 ? 256 : 128;
}

int32_t launch_update(const void* q, const void* k, const void* v, float* m, float* l, float* acc,
                      int64_t sq_t, int64_t sq_h, int64_t sk_t, int64_t sk_h, int64_t sv_t,
                      int64_t sv_h, int64_t ss_t, int64_t ss_h, int64_t sa_t, int64_t sa_h,
                      int32_t q_tokens, int32_t kv_tokens, int32_t q_heads, int32_t kv_heads,
                      int32_t head_dim, int32_t q_local_offset, int32_t kv_local_offset,
                      int32_t causal_shift, double softmax_scale, int32_t flags, int32_t dtype,
                      hipStream_t stream, int32_t merge_keys, const FusedOutput* fused,
                      bool v_transposed, bool tiled_state) {
  if (dtype != SA_DTYPE_BF16 && dtype != SA_DTYPE_FP16) {
    set_error("sa_update_attention_state: unsupported dtype code %d", dtype);
    return SA_ERR_UNSUPPORTED_DTYPE;
  }
  if (head_dim < 16 || head_dim > 256 || head_dim % 8 != 0) {
    set_error("sa_update_attention_state: head_dim must be a multiple of 8 in [16, 256], got %d",
              head_dim);
    return SA_ERR_UNSUPPORTED_HEAD_DIM;
  }
  if (q_tokens < 0 || kv_tokens < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0) {
    set_error("sa_update_attention_state: bad sizes q_tokens=%d kv_tokens=%d q_heads=%d kv_heads=%d",
              q_tokens, kv_tokens, q_heads, kv_heads);
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (q_tokens == 0) return 0;
  // A fused launch writes the output instead of the state; one that also
  // initializes the state does not touch m, l and acc, which may be null.
  const bool starts_state = (flags & SA_FLAG_INITIALIZE) != 0;
  if (!q || !k || !v || (!(fused != nullptr && starts_state) && (!m || !l || !acc))) {
    set_error("sa_update_attention_state: null pointer argument");
    return SA_ERR_INVALID_ARGUMENT;
  }
  // 16-byte vector access of 8 elements (inputs) and 4 floats (accumulator).
  const int64_t el_strides[] = {sq_t, sq_h, sk_t, sk_h, sv_t, sv_h};
  for (int64_t st : el_strides) {
    if (st % 8 != 0) {
      set_error("sa_update_attention_state: q/k/v token and head strides must be multiples of 8 elements");
      return SA_ERR_INVALID_ARGUMENT;
    }
  }
  if (sk_t <= 0 || sv_t <= 0 || sk_t >= (1 << 24) || sv_t >= (1 << 24)) {
    // Per-lane offsets within a 64-key tile are 32-bit.
    set_error("sa_update_attention_state: k/v token strides must be in [1, 2^24) elements");
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (sa_t % 4 != 0 || sa_h % 4 != 0 || !aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) ||
      !aligned(acc, 16) || !aligned(m, 4) || !aligned(l, 4)) {
    set_error("sa_update_attention_state: buffers must be 16-byte aligned with vector-aligned strides");
    return SA_ERR_INVALID_ARGUMENT;
  }
  UpdateParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.m = m;
  p.l = l;
  p.acc = acc;
  p.sq_t = sq_t; p.sq_h = sq_h; p.sk_t = sk_t; p.sk_h = sk_h; p.sv_t = sv_t; p.sv_h = sv_h;
  p.ss_t = ss_t; p.ss_h = ss_h; p.sa_t = sa_t; p.sa_h = sa_h;
  p.q_tokens = q_tokens;
  p.kv_tokens = kv_tokens;
  p.group = q_heads / kv_heads;
  p.head_dim = head_dim;
  p.q_local_offset = q_local_offset;
  p.kv_local_offset = kv_local_offset;
  p.causal_shift = causal_shift;
  p.scale_log2 = (float)(softmax_scale * 1.4426950408889634);
  if (merge_keys < 0 || merge_keys % 64 != 0) {
    set_error("merge_keys %d is not a multiple of the 64-key tile", merge_keys);
    return SA_ERR_INVALID_ARGUMENT;
  }
  p.merge_tiles = merge_keys / 64;
  p.tiled_state = tiled_state ? 1 : 0;
  if (fused != nullptr) {
    // Same output layout rules as the finalize kernel.
    if (!fused->out || fused->so_t % 8 != 0 || fused->so_h % 8 != 0 || !aligned(fused->out, 16)) {
      set_error("fused finalize needs a 16-byte aligned output with vector-aligned strides");
      return SA_ERR_INVALID_ARGUMENT;
    }
    p.out = static_cast<uint16_t*>(fused->out);
    p.so_t = fused->so_t;
    p.so_h = fused->so_h;
    p.lse = fused->lse;
    p.lse_sh = fused->lse_sh;
    p.lse_off = fused->lse_off;
  }
  // Workgroup numbering is 32-bit: at least 128 queries per workgroup.
  int64_t longest_q = fused != nullptr && fused->num_segments > 0 ? 0 : q_tokens;
  for (int32_t s = 0; fused != nullptr && s < fused->num_segments; ++s)
    longest_q = std::max<int64_t>(longest_q, fused->segments[s].q_len);
  if ((longest_q + 127) / 128 * q_heads > (int64_t)INT32_MAX / 8) {
    set_error("sa_update_attention_state: q_tokens * q_heads too large for one launch");
    return SA_ERR_INVALID_ARGUMENT;
  }
  p.q_heads = q_heads;
  p.causal = (flags & SA_FLAG_CAUSAL) != 0;
  p.init = starts_state;
  // V transposed: v is transpose_v_kernel's layout, row stride sv_t (keys
  // padded to whole 64-key tiles), head stride sv_h.
  if (v_transposed && (head_dim != 128 || !starts_state || sv_t % 64 != 0 || sv_t < kv_tokens || sv_h < 128 * sv_t)) {
    set_error("transposed V needs head_dim 128, an initializing launch and a padded [heads][128][keys] layout");
    return SA_ERR_INVALID_ARGUMENT;
  }
  const bool overlapped = (flags & kLaunchOverlapped) != 0;
  if (fused != nullptr && fused->num_segments > 0) {
    if (v_transposed || !starts_state) {
      set_error("a launch over segments reads V in place and loads no state");
      return SA_ERR_INVALID_ARGUMENT;
    }
    return launch_segments(p, *fused, dtype, overlapped, stream);
  }
  const hipError_t err = launch_update_variant(p, v_transposed ? kTransposedV : kRows, dtype, overlapped, stream);
  return err == hipSuccess ? 0 : hip_status(err, "update kernel launch");
}

int32_t launch_update_int8(const void* q, const void* k, const void* v, const void* k_scales,
                           const void* v_scales, float* m, float* l, float* acc, int64_t sq_t,
                           int64_t sq_h, int64_t sk_t, int64_t sk_h, int64_t sv_t, int64_t sv_h,
                           int64_t sks_g, int64_t sks_h, int64_t svs_g, int64_t svs_h,
                           int64_t ss_t, int64_t ss_h, int64_t sa_t, int64_t sa_h,
                           int32_t q_tokens, int32_t kv_tokens, int32_t q_heads, int32_t kv_heads,
                           int32_t head_dim, int32_t q_local_offset, int32_t kv_local_offset,
                           int32_t storage_token_offset, int32_t causal_shift,
                           double softmax_scale, int32_t flags, int32_t dtype,
                           int32_t quant_group_tokens, hipStream_t stream, bool tiled_state) {
  if (dtype != SA_DTYPE_BF16 && dtype != SA_DTYPE_FP16) {
    set_error("sa_update_attention_state_int8: unsupported query dtype code %d", dtype);
    return SA_ERR_UNSUPPORTED_DTYPE;
  }
  if (head_dim < 16 || head_dim > 128 || head_dim % 16 != 0) {
    set_error("sa_update_attention_state_int8: head_dim must be a multiple of 16 in [16, 128], got %d",
              head_dim);
    return SA_ERR_UNSUPPORTED_HEAD_DIM;
  }
  if (q_tokens < 0 || kv_tokens < 0 || q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 ||
      storage_token_offset < 0) {
    set_error("sa_update_attention_state_int8: bad sizes q_tokens=%d kv_tokens=%d q_heads=%d kv_heads=%d "
              "storage_token_offset=%d", q_tokens, kv_tokens, q_heads, kv_heads, storage_token_offset);
    return SA_ERR_INVALID_ARGUMENT;
  }
  int shift = 0;
  while (shift < 30 && (1 << shift) < quant_group_tokens) ++shift;
  if (quant_group_tokens <= 0 || (1 << shift) != quant_group_tokens) {
    set_error("sa_update_attention_state_int8: quant_group_tokens must be a power of two, got %d",
              quant_group_tokens);
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (q_tokens == 0) return 0;
  if (!q || !k || !v || !k_scales || !v_scales || !m || !l || !acc) {
    set_error("sa_update_attention_state_int8: null pointer argument");
    return SA_ERR_INVALID_ARGUMENT;
  }
  // Q: 16-byte vectors of 8 elements; int8 K/V: 16-byte DMA granules.
  if (sq_t % 8 != 0 || sq_h % 8 != 0 || sk_t % 16 != 0 || sk_h % 16 != 0 || sv_t % 16 != 0 ||
      sv_h % 16 != 0) {
    set_error("sa_update_attention_state_int8: q strides must be multiples of 8 elements and int8 "
              "k/v strides multiples of 16");
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (sk_t <= 0 || sv_t <= 0 || sk_t >= (1 << 24) || sv_t >= (1 << 24)) {
    set_error("sa_update_attention_state_int8: k/v token strides must be in [1, 2^24) elements");
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (sa_t % 4 != 0 || sa_h % 4 != 0 || !aligned(q, 16) || !aligned(k, 16) || !aligned(v, 16) ||
      !aligned(acc, 16) || !aligned(m, 4) || !aligned(l, 4) || !aligned(k_scales, 2) ||
      !aligned(v_scales, 2)) {
    set_error("sa_update_attention_state_int8: buffers must be aligned (16 bytes for q/k/v/acc, 2 for scales)");
    return SA_ERR_INVALID_ARGUMENT;
  }
  UpdateParams p{};
  p.q = static_cast<const uint16_t*>(q);
  p.k = static_cast<const uint16_t*>(k);
  p.v = static_cast<const uint16_t*>(v);
  p.m = m;
  p.l = l;
  p.acc = acc;
  p.sq_t = sq_t; p.sq_h = sq_h; p.sk_t = sk_t; p.sk_h = sk_h; p.sv_t = sv_t; p.sv_h = sv_h;
  p.ss_t = ss_t; p.ss_h = ss_h; p.sa_t = sa_t; p.sa_h = sa_h;
  p.q_tokens = q_tokens;
  p.kv_tokens = kv_tokens;
  p.group = q_heads / kv_heads;
  p.head_dim = head_dim;
  p.q_local_offset = q_local_offset;
  p.kv_local_offset = kv_local_offset;
  p.causal_shift = causal_shift;
  p.scale_log2 = (float)(softmax_scale * 1.4426950408889634);
  p.q_heads = q_heads;
  p.ks = static_cast<const uint16_t*>(k_scales);
  p.vs = static_cast<const uint16_t*>(v_scales);
  p.sks_g = sks_g; p.sks_h = sks_h; p.svs_g = svs_g; p.svs_h = svs_h;
  p.scale_offset = storage_token_offset;
  p.scale_shift = shift;
  p.tiled_state = tiled_state ? 1 : 0;
  p.causal = (flags & SA_FLAG_CAUSAL) != 0;
  p.init = (flags & SA_FLAG_INITIALIZE) != 0;
  const hipError_t err = launch_update_variant(p, kInt8, dtype, false, stream);
  return err == hipSuccess ? 0 : hip_status(err, "int8 update kernel launch");
}

int32_t launch_transpose_v(const void* v, int64_t sv_t, int64_t sv_h, int32_t kv_tokens, int32_t kv_heads,
                           int32_t head_dim, void* vt, int64_t t_pad, hipStream_t stream) {
  if (head_dim != 128 || kv_tokens < 0 || kv_heads <= 0 || t_pad % 64 != 0 || t_pad < kv_tokens ||
      t_pad >= (1 << 24) || !v || !vt || sv_t % 8 != 0 || sv_h % 8 != 0 || !aligned(v, 16) ||
      !aligned(vt, 16)) {
    set_error("transpose of V: bad arguments (head_dim %d, kv_tokens %d, kv_heads %d, padded keys %lld)",
              head_dim, kv_tokens, kv_heads, (long long)t_pad);
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (t_pad == 0) return 0;
  TransposeParams p;
  p.v = static_cast<const uint16_t*>(v);
  p.vt = static_cast<uint16_t*>(vt);
  p.sv_t = sv_t;
  p.sv_h = sv_h;
  p.t_pad = t_pad;
  p.kv_tokens = kv_tokens;
  p.tiles = (int32_t)(t_pad / 64);
  hipLaunchKernelGGL(transpose_v_kernel, dim3((unsigned)((int64_t)kv_heads * p.tiles)), dim3(256), 0, stream, p);
  const hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_status(err, "transpose of V");
}

int32_t launch_finalize(const float* acc, const float* m, const float* l, void* out, float* lse,
                        int64_t sa_t, int64_t sa_h, int64_t ss_t, int64_t ss_h, int64_t so_t,
                        int64_t so_h, int64_t lse_sh, int64_t lse_off, int32_t q_tokens,
                        int32_t q_heads, int32_t head_dim, int32_t dtype, hipStream_t stream,
                        bool tiled_state) {
  if (dtype != SA_DTYPE_BF16 && dtype != SA_DTYPE_FP16) {
    set_error("sa_finalize_attention: unsupported dtype code %d", dtype);
    return SA_ERR_UNSUPPORTED_DTYPE;
  }
  if (head_dim < 8 || head_dim > 256 || head_dim % 8 != 0) {
    set_error("sa_finalize_attention: head_dim must be a multiple of 8 in [8, 256], got %d", head_dim);
    return SA_ERR_UNSUPPORTED_HEAD_DIM;
  }
  if (q_tokens < 0 || q_heads <= 0) {
    set_error("sa_finalize_attention: bad sizes q_tokens=%d q_heads=%d", q_tokens, q_heads);
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (q_tokens == 0) return 0;
  if (!acc || !l || !out || (lse && !m)) {
    set_error("sa_finalize_attention: null pointer argument");
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (sa_t % 4 != 0 || sa_h % 4 != 0 || so_t % 8 != 0 || so_h % 8 != 0 || !aligned(acc, 16) ||
      !aligned(out, 16)) {
    set_error("sa_finalize_attention: buffers must be 16-byte aligned with vector-aligned strides");
    return SA_ERR_INVALID_ARGUMENT;
  }
  FinalizeParams p;
  p.acc = acc;
  p.m = m;
  p.l = l;
  p.out = static_cast<uint16_t*>(out);
  p.lse = lse;
  p.sa_t = sa_t; p.sa_h = sa_h; p.ss_t = ss_t; p.ss_h = ss_h; p.so_t = so_t; p.so_h = so_h;
  p.lse_sh = lse_sh;
  p.lse_off = lse_off;
  p.groups = head_dim / 8;
  p.q_tokens = q_tokens;
  p.q_heads = q_heads;
  p.tiled_state = tiled_state ? 1 : 0;
  if (q_heads > 65535) {
    set_error("sa_finalize_attention: q_heads %d exceeds the grid's 65,535 heads", q_heads);
    return SA_ERR_INVALID_ARGUMENT;
  }
  const dim3 grid((unsigned)(((int64_t)q_tokens + 15) / 16), (unsigned)q_heads);
  if (dtype == SA_DTYPE_BF16)
    hipLaunchKernelGGL(finalize_kernel<BF16>, grid, dim3(256), 0, stream, p);
  else
    hipLaunchKernelGGL(finalize_kernel<FP16>, grid, dim3(256), 0, stream, p);
  hipError_t err = hipGetLastError();
  return err == hipSuccess ? 0 : hip_status(err, "finalize kernel launch");
}

}  // namespace sa

namespace {

// Device scratch of sa_run_resident_noalloc: the transposed copy of V that
// the resident update launch reads.  One array per GPU, held from the first
// load of this library's code object until the process ends.  In host code
// the name is only a stand-in for the symbol: the array's address on a
// device comes from hipGetSymbolAddress with that device current, looked up
// once per device and kept below.
constexpr int64_t kNoAllocScratchBytes = int64_t(64) << 20;
constexpr int kMaxDevices = 64;
__device__ __align__(256) uint8_t scratch[kNoAllocScratchBytes];

std::mutex g_scratch_mutex;
void* g_scratch_address[kMaxDevices] = {};

int32_t scratch_on_current_device(void** address) {
  int device = 0;
  hipError_t err = hipGetDevice(&device);
  if (err != hipSuccess) return sa::hip_status(err, "sa_run_resident_noalloc: hipGetDevice");
  if (device < 0 || device >= kMaxDevices) {
    sa::set_error("sa_run_resident_noalloc: device ordinal %d outside [0, %d)", device, kMaxDevices);
    return SA_ERR_BAD_STATE;
  }
  std::lock_guard<std::mutex> lock(g_scratch_mutex);
  if (g_scratch_address[device] == nullptr) {
    void* found = nullptr;
    err = hipGetSymbolAddress(&found, HIP_SYMBOL(scratch));
    if (err != hipSuccess) return sa::hip_status(err, "sa_run_resident_noalloc: hipGetSymbolAddress(scratch)");
    if (found == nullptr || reinterpret_cast<uintptr_t>(found) % 256 != 0) {
      sa::set_error("sa_run_resident_noalloc: scratch address %p is not 256-byte aligned", found);
      return SA_ERR_BAD_STATE;
    }
    g_scratch_address[device] = found;
  }
  *address = g_scratch_address[device];
  return 0;
}

}  // namespace

extern "C" {

int32_t sa_update_launch_shape(const int32_t* q_tokens, const int32_t* kv_tokens, int32_t num_segments,
                               int32_t q_heads, int32_t kv_heads, int32_t head_dim, int32_t causal_shift,
                               int32_t causal, int32_t kv_layout, int32_t overlapped, int32_t* rows, int32_t* stages,
                               int64_t* workgroups) {
  sa::clear_error();
  if (!q_tokens || !kv_tokens || num_segments < 1 || num_segments > sa::kMaxSegments || q_heads <= 0 ||
      kv_heads <= 0 || q_heads % kv_heads != 0 || head_dim < 16 || head_dim > 256 || kv_layout < sa::kRows ||
      kv_layout > sa::kInt8 || (kv_layout == sa::kTransposedV && head_dim != 128) ||
      (kv_layout == sa::kInt8 && head_dim > 128) || (kv_layout != sa::kRows && num_segments > 1) || !rows || !stages ||
      !workgroups) {
    sa::set_error("sa_update_launch_shape: bad argument");
    return SA_ERR_INVALID_ARGUMENT;
  }
  sa::UpdateParams p{};
  p.q_heads = q_heads;
  p.group = q_heads / kv_heads;
  p.head_dim = head_dim;
  p.causal = causal != 0;
  p.causal_shift = causal_shift;
  p.q_tokens = q_tokens[0];
  p.kv_tokens = kv_tokens[0];
  p.segments = num_segments > 1 ? num_segments : 0;
  for (int32_t s = 0; s < num_segments; ++s) {
    if (q_tokens[s] <= 0 || kv_tokens[s] < 0 || ((int64_t)q_tokens[s] + 127) / 128 * q_heads > INT32_MAX / 256) {
      sa::set_error("sa_update_launch_shape: segment %d has bad sizes", s);
      return SA_ERR_INVALID_ARGUMENT;
    }
    p.segment[s] = sa::Segment{0, 0, q_tokens[s], kv_tokens[s]};
  }
  const sa::LaunchShape shape = sa::shape_launch(p, kv_layout, overlapped != 0);
  *rows = shape.rows;
  *stages = shape.stages;
  *workgroups = shape.grid;
  return 0;
}

int32_t sa_run_resident_noalloc(const void* q, const void* k, const void* v, void* out, float* lse,
                                int64_t stride_qt, int64_t stride_qh, int64_t stride_kt,
                                int64_t stride_kh, int64_t stride_vt, int64_t stride_vh,
                                int64_t stride_ot, int64_t stride_oh, int64_t lse_stride_h,
                                const int64_t* cu_seqlens_q, const int64_t* cu_seqlens_k,
                                int32_t num_segments, int32_t q_heads, int32_t kv_heads,
                                int32_t head_dim, int32_t dtype, int32_t kv_chunk_tokens,
                                double softmax_scale, int32_t causal, void* stream) try {
  sa::clear_error();
  if (!q || !k || !v || !out || !cu_seqlens_q || !cu_seqlens_k || num_segments < 0) {
    sa::set_error("sa_run_resident_noalloc: null argument");
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (head_dim != 128) {
    sa::set_error("sa_run_resident_noalloc: the transposed-V launch needs head_dim 128, got %d", head_dim);
    return SA_ERR_UNSUPPORTED_HEAD_DIM;
  }
  if (dtype != SA_DTYPE_BF16 && dtype != SA_DTYPE_FP16) {
    sa::set_error("sa_run_resident_noalloc: unsupported dtype code %d", dtype);
    return SA_ERR_UNSUPPORTED_DTYPE;
  }
  if (q_heads <= 0 || kv_heads <= 0 || q_heads % kv_heads != 0 || kv_chunk_tokens <= 0 ||
      kv_chunk_tokens % 64 != 0) {
    sa::set_error("sa_run_resident_noalloc: bad heads %d/%d or K/V chunk %d (a positive multiple of 64)",
                  q_heads, kv_heads, kv_chunk_tokens);
    return SA_ERR_INVALID_ARGUMENT;
  }
  if (stride_ot % 8 != 0 || stride_oh % 8 != 0 || !sa::aligned(out, 16)) {
    sa::set_error("sa_run_resident_noalloc: out must be 16-byte aligned with strides that are multiples of 8");
    return SA_ERR_INVALID_ARGUMENT;
  }
  // The launches' own argument rules, checked here so that a call they would
  // reject is rejected before anything is enqueued on the shared scratch.
  const int64_t in_strides[] = {stride_qt, stride_qh, stride_kt, stride_kh, stride_vt, stride_vh};
  for (int64_t st : in_strides) {
    if (st % 8 != 0) {
      sa::set_error("sa_run_resident_noalloc: q/k/v token and head strides must be multiples of 8 elements");
      return SA_ERR_INVALID_ARGUMENT;
    }
  }
  if (stride_kt <= 0 || stride_kt >= (1 << 24) || !sa::aligned(q, 16) || !sa::aligned(k, 16) || !sa::aligned(v, 16) ||
      (lse != nullptr && !sa::aligned(lse, 4))) {
    sa::set_error("sa_run_resident_noalloc: q/k/v must be 16-byte aligned (lse 4-byte) and the k token stride "
                  "in [1, 2^24) elements");
    return SA_ERR_INVALID_ARGUMENT;
  }
  // Every segment is checked before anything is enqueued.
  for (int32_t s = 0; s < num_segments; ++s) {
    const int64_t q_length = cu_seqlens_q[s + 1] - cu_seqlens_q[s];
    const int64_t k_length = cu_seqlens_k[s + 1] - cu_seqlens_k[s];
    if (q_length < 0 || k_length < 0 || (q_length > 0 && k_length == 0) || q_length > INT32_MAX ||
        k_length >= (1 << 24)) {
      sa::set_error("sa_run_resident_noalloc: segment %d has invalid bounds", s);
      return SA_ERR_INVALID_ARGUMENT;
    }
    // Workgroup numbering of the update launch is 32-bit.
    if ((q_length + 127) / 128 * q_heads > (int64_t)INT32_MAX / 8) {
      sa::set_error("sa_run_resident_noalloc: segment %d has too many queries x heads for one launch", s);
      return SA_ERR_INVALID_ARGUMENT;
    }
    const int64_t needed = (int64_t)kv_heads * 128 * ((k_length + 63) / 64 * 64) * 2;
    if (q_length > 0 && needed > kNoAllocScratchBytes) {
      sa::set_error("sa_run_resident_noalloc: segment %d needs %lld bytes of transposed-V scratch; this entry "
                    "point has %lld (kv_heads * 128 * keys rounded up to 64 * 2 bytes per segment)",
                    s, (long long)needed, (long long)kNoAllocScratchBytes);
      return SA_ERR_INVALID_ARGUMENT;
    }
  }
  void* vt = nullptr;
  int32_t rc = scratch_on_current_device(&vt);
  if (rc != 0) return rc;
  hipStream_t hs = static_cast<hipStream_t>(stream);
  const char* qd = static_cast<const char*>(q);
  const char* kd = static_cast<const char*>(k);
  const char* vd = static_cast<const char*>(v);
  char* od = static_cast<char*>(out);
  // The launch sequence of sa_pipeline_run_resident's fused path with the
  // scratch in place of the attached one: per segment of enough queries V
  // transposed (zero keys up to the 64-key tile), then one update launch over
  // it that finalizes in its epilogue with the row sums merged at every K/V
  // chunk boundary; the other segments together.  All launches are on
  // `stream`, so a later segment's transpose starts after this segment's
  // update has read the scratch.
  const auto launch = [&](const char* v_seg, int64_t sv_t, int64_t sv_h, int64_t q_start, int64_t q_length,
                          int64_t k_start, int64_t k_length, const sa::FusedOutput& fused, bool transposed) {
    return sa::launch_update(qd + q_start * stride_qt * 2, kd + k_start * stride_kt * 2, v_seg, nullptr, nullptr,
                             nullptr, stride_qt, stride_qh, stride_kt, stride_kh, sv_t, sv_h, 0, 0, 0, 0,
                             (int32_t)q_length, (int32_t)k_length, q_heads, kv_heads, 128, 0, 0,
                             (int32_t)(k_length - q_length), softmax_scale,
                             (causal ? SA_FLAG_CAUSAL : 0) | SA_FLAG_INITIALIZE, dtype, hs, kv_chunk_tokens, &fused,
                             transposed);
  };
  sa::SegmentGroup together;
  for (int32_t s = 0; s < num_segments; ++s) {
    const int64_t q_start = cu_seqlens_q[s], k_start = cu_seqlens_k[s];
    const int64_t q_length = cu_seqlens_q[s + 1] - q_start, k_length = cu_seqlens_k[s + 1] - k_start;
    if (q_length == 0) continue;
    if (!sa::transposes_v(q_length, q_heads / kv_heads, stride_vt) && together.add(q_start, q_length, k_start, k_length)) continue;
    const int64_t t_pad = (k_length + 63) / 64 * 64;
    rc = sa::launch_transpose_v(vd + k_start * stride_vt * 2, stride_vt, stride_vh, (int32_t)k_length, kv_heads, 128,
                                vt, t_pad, hs);
    if (rc != 0) return rc;
    const sa::FusedOutput fused{od + q_start * stride_ot * 2, stride_ot, stride_oh, lse, lse_stride_h, q_start};
    rc = launch(static_cast<const char*>(vt), t_pad, 128 * t_pad, q_start, q_length, k_start, k_length, fused, true);
    if (rc != 0) return rc;
  }
  if (together.segments.empty()) return 0;
  const sa::FusedOutput fused{od + together.q0 * stride_ot * 2, stride_ot, stride_oh, lse, lse_stride_h, together.q0,
                              together.segments.data(), (int32_t)together.segments.size()};
  return launch(vd + together.k0 * stride_vt * 2, stride_vt, stride_vh, together.q0, together.q_span(), together.k0,
                together.k_span(), fused, false);
} catch (const std::exception& error) {
  return sa::exception_status("sa_run_resident_noalloc", error);
}

int32_t sa_update_attention_state(const void* q, const void* k, const void* v, float* running_max,
                                  float* running_sum, float* accumulator, int64_t stride_qt,
                                  int64_t stride_qh, int64_t stride_kt, int64_t stride_kh,
                                  int64_t stride_vt, int64_t stride_vh, int64_t stride_st,
                                  int64_t stride_sh, int64_t stride_at, int64_t stride_ah,
                                  int32_t q_tokens, int32_t kv_tokens, int32_t q_heads,
                                  int32_t kv_heads, int32_t head_dim, int32_t q_local_offset,
                                  int32_t kv_local_offset, int32_t causal_shift,
                                  double softmax_scale, int32_t flags, int32_t dtype, void* stream) {
  sa::clear_error();
  return sa::launch_update(q, k, v, running_max, running_sum, accumulator, stride_qt, stride_qh,
                           stride_kt, stride_kh, stride_vt, stride_vh, stride_st, stride_sh,
                           stride_at, stride_ah, q_tokens, kv_tokens, q_heads, kv_heads, head_dim,
                           q_local_offset, kv_local_offset, causal_shift, softmax_scale,
                           flags & (SA_FLAG_CAUSAL | SA_FLAG_INITIALIZE), dtype, static_cast<hipStream_t>(stream));
}

int32_t sa_update_attention_state_int8(
    const void* q, const void* k, const void* v, const void* k_scales, const void* v_scales,
    float* running_max, float* running_sum, float* accumulator, int64_t stride_qt,
    int64_t stride_qh, int64_t stride_kt, int64_t stride_kh, int64_t stride_vt, int64_t stride_vh,
    int64_t stride_ksg, int64_t stride_ksh, int64_t stride_vsg, int64_t stride_vsh,
    int64_t stride_st, int64_t stride_sh, int64_t stride_at, int64_t stride_ah, int32_t q_tokens,
    int32_t kv_tokens, int32_t q_heads, int32_t kv_heads, int32_t head_dim, int32_t q_local_offset,
    int32_t kv_local_offset, int32_t storage_token_offset, int32_t causal_shift,
    double softmax_scale, int32_t flags, int32_t dtype, int32_t quant_group_tokens, void* stream) {
  sa::clear_error();
  return sa::launch_update_int8(q, k, v, k_scales, v_scales, running_max, running_sum, accumulator,
                                stride_qt, stride_qh, stride_kt, stride_kh, stride_vt, stride_vh,
                                stride_ksg, stride_ksh, stride_vsg, stride_vsh, stride_st, stride_sh,
                                stride_at, stride_ah, q_tokens, kv_tokens, q_heads, kv_heads,
                                head_dim, q_local_offset, kv_local_offset, storage_token_offset,
                                causal_shift, softmax_scale, flags, dtype, quant_group_tokens,
                                static_cast<hipStream_t>(stream));
}

int32_t sa_finalize_attention(const float* accumulator, const float* running_max,
                              const float* running_sum, void* out, float* lse, int64_t stride_at,
                              int64_t stride_ah, int64_t stride_st, int64_t stride_sh,
                              int64_t stride_ot, int64_t stride_oh, int64_t lse_stride_h,
                              int64_t lse_token_offset, int32_t q_tokens, int32_t q_heads,
                              int32_t head_dim, int32_t dtype, void* stream) {
  sa::clear_error();
  return sa::launch_finalize(accumulator, running_max, running_sum, out, lse, stride_at, stride_ah,
                             stride_st, stride_sh, stride_ot, stride_oh, lse_stride_h,
                             lse_token_offset, q_tokens, q_heads, head_dim, dtype,
                             static_cast<hipStream_t>(stream));
}

}  // extern "C"
