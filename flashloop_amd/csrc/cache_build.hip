// Host-side set-up of a packed cache as device passes: what CrossLoopKVLayer.from_prefill and
// its rollover do around fl_pack_kv_groups (flashloop/cache.py:752-817, 1778-1838).
//
//  * fl_count_active_rows -- rows of streams 2/3 a prefill's masks keep, and whether the masks
//    are nested.
//  * fl_cache_prepare -- one launch over the parts of a new layer that the pack kernel does not
//    write: lengths, rank maps, BF16 tails and their activity, zeros in the unused capacity.
//  * fl_roll_begin / fl_roll_end -- the rank-map rows of a rolled-out group before it is
//    packed, and the tail's shift and the lengths after.
//
// All are bound by their launch or by the bytes they write.  As torch ops a build was 91 to 176
// launches and three host synchronisations (layer of 16 heads, 8192 tokens, masked: 653 us, of
// which the pack kernel took 83; now 152, one synchronisation) and a rollover ~40 launches (a
// ragged batch of eight over four layers: 1324 us a token before, 1253 now).
#include <algorithm>

#include "fl_common.h"

namespace fl {
namespace {

constexpr int kBuildThreads = 512;
constexpr int kBuildWaves = kBuildThreads / kWave;
constexpr int kMaxSeqs = 64;      // most sequences of one launch (their lengths travel as arguments)
constexpr int kScanPer = 16;      // tokens per thread and scan step
constexpr int kClearBytes = 32768;  // per workgroup
constexpr int kRegions = 21;

struct Lengths {
  int32_t packed[kMaxSeqs];
  int32_t tail[kMaxSeqs];
  int32_t late[2][kMaxSeqs];
};

// Exclusive prefix of v over the workgroup; *total receives the sum.
__device__ __forceinline__ int block_prefix(int v, int* sh, int* total) {
  const int lane = threadIdx.x & 63, w = threadIdx.x >> 6;
  int incl = v;
#pragma unroll
  for (int off = 1; off < kWave; off <<= 1) {
    const int o = __shfl_up(incl, off, kWave);
    if (lane >= off) incl += o;
  }
  __syncthreads();
  if (lane == 63) sh[w] = incl;
  __syncthreads();
  int before = 0, sum = 0;
#pragma unroll
  for (int i = 0; i < kBuildWaves; ++i) {
    if (i < w) before += sh[i];
    sum += sh[i];
  }
  *total = sum;
  return before + incl - v;
}

// Bit e: token t0 + e is below n and active (null mask: every token is).
__device__ __forceinline__ uint32_t active_bits(const uint8_t* mask, int t0, int n) {
  uint32_t bits = 0;
  if (mask == nullptr) {
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) bits |= t0 + e < n ? 1u << e : 0u;
  } else {
    uint8_t m[kScanPer];
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) m[e] = mask[max(0, min(t0 + e, n - 1))];
#pragma unroll
    for (int e = 0; e < kScanPer; ++e) bits |= (t0 + e < n && m[e] != 0) ? 1u << e : 0u;
  }
  return bits;
}

// Workgroup (b, s): active tokens of mask s below the sequence's packed prefix; the s = 1
// workgroups also look for a token of mask 1 that mask 0 leaves out, over every token.
__global__ __launch_bounds__(kBuildThreads) void count_active_kernel(const uint8_t* mask0, const uint8_t* mask1,
                                                                     int64_t stride, int tokens, Lengths len, int b0,
                                                                     int batch, int32_t* counts) {
  __shared__ int sh[kBuildWaves];
  const int i = blockIdx.x, s = blockIdx.y, b = b0 + i;
  const uint8_t* m0 = mask0 ? mask0 + b * stride : nullptr;
  const uint8_t* m1 = mask1 ? mask1 + b * stride : nullptr;
  const int n = len.packed[i];
  int count = 0, bad = 0;
  for (int base = 0; base < tokens; base += kBuildThreads * kScanPer) {
    const int t0 = base + static_cast<int>(threadIdx.x) * kScanPer;
    if (t0 >= tokens) continue;
    const uint32_t a = active_bits(s == 0 ? m0 : m1, t0, tokens);
    if (s == 1) bad |= (a & ~active_bits(m0, t0, tokens)) != 0u;
    const int in = n - t0;  // tokens of the chunk below the prefix
    count += __popc(in >= kScanPer ? a : (in > 0 ? a & ((1u << in) - 1u) : 0u));
  }
  int total;
  block_prefix(count, sh, &total);
  if (threadIdx.x == 0) counts[s * batch + b] = total;
  if (bad) atomicOr(&counts[2 * batch], 1);
}

// One of the layer's buffers as bytes: rows of `row` bytes per (b,h), `unit` bytes per token,
// 64-token group or compact row of it.
struct Region {
  uint8_t* base;
  int64_t row;
  int32_t unit;
  int32_t kind;  // used units: 0 packed tokens, 1 packed groups, 2 / 3 compact rows of streams 2 / 3
};

struct PrepareArgs {
  fl_cache_view v;
  int b0, seqs;
  int64_t src_stride, mask_stride;
  const uint16_t* src[8];  // K of loops 1..4, then V
  const uint8_t* mask[2];
  uint8_t* tail_active[2];
  int32_t* packed_tokens;
  int32_t* tail_tokens;
  int32_t* late_rows;   // [2, B]
  int32_t* dst_group0;  // [B], zeroed
  Region region[kRegions];
  int clear_chunks;  // workgroups per (b,h) and region
  Lengths len;
};

// Workgroup ranges: rank maps (2 per sequence), tail activity and lengths (1 per sequence),
// tails (8 per (b,h)), then the clears.
__global__ __launch_bounds__(kBuildThreads) void cache_prepare_kernel(PrepareArgs a) {
  __shared__ int sh[kBuildWaves];
  const fl_cache_view& v = a.v;
  int blk = blockIdx.x;
  const int tid = threadIdx.x;
  if (blk < 2 * a.seqs) {
    const int s = blk / a.seqs, i = blk % a.seqs, b = a.b0 + i;
    const int n = a.len.packed[i], cap = v.token_capacity, rows = a.len.late[s][i];  // (a rollover goes on from there)
    const uint8_t* m = a.mask[s] ? a.mask[s] + b * a.mask_stride : nullptr;
    int32_t* out = v.rank[s] + static_cast<int64_t>(b) * cap;
    int run = 0;
    for (int base = 0; base < cap; base += kBuildThreads * kScanPer) {
      const int t0 = base + tid * kScanPer;
      const uint32_t bits = t0 < n ? active_bits(m, t0, n) : 0u;
      int total;
      int r = run + block_prefix(__popc(bits), sh, &total);
      run += total;
      if (t0 < cap) {
#pragma unroll
        for (int q = 0; q < kScanPer / 4; ++q) {
          int x[4];
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            const bool on = (bits >> (4 * q + e)) & 1u;
            x[e] = on && r < rows ? r : -1;
            r += on ? 1 : 0;
          }
          *reinterpret_cast<int4*>(out + t0 + 4 * q) = make_int4(x[0], x[1], x[2], x[3]);
        }
      }
    }
    return;
  }
  blk -= 2 * a.seqs;
  if (blk < a.seqs) {
    const int i = blk, b = a.b0 + i;
    if (tid == 0) {
      a.packed_tokens[b] = a.len.packed[i];
      a.tail_tokens[b] = a.len.tail[i];
      a.late_rows[b] = a.len.late[0][i];
      a.late_rows[v.batch + b] = a.len.late[1][i];
      a.dst_group0[b] = 0;
    }
#pragma unroll
    for (int s = 0; s < 2; ++s)
      for (int r = tid; r < v.tail_capacity; r += kBuildThreads)
        a.tail_active[s][static_cast<int64_t>(b) * v.tail_capacity + r] =
            r < a.len.tail[i] && (a.mask[s] == nullptr || a.mask[s][b * a.mask_stride + a.len.packed[i] + r] != 0);
    return;
  }
  blk -= a.seqs;
  const int rows = a.seqs * v.heads;
  if (blk < 8 * rows) {
    const int t = blk / rows, bh = a.b0 * v.heads + blk % rows, i = (blk % rows) / v.heads;
    uint16_t* dst = nullptr;
    const uint16_t* src = nullptr;
#pragma unroll
    for (int k = 0; k < 8; ++k)
      if (k == t) {
        dst = k < 4 ? v.tail_key[k & 3] : v.tail_value[k & 3];
        src = a.src[k];
      }
    dst += static_cast<int64_t>(bh) * v.tail_capacity * kDim;
    src += (static_cast<int64_t>(bh) * a.src_stride + a.len.packed[i]) * kDim;
    const int live = a.len.tail[i] * (kDim / 8), all = v.tail_capacity * (kDim / 8);
    for (int c = tid; c < all; c += kBuildThreads)
      reinterpret_cast<uint4*>(dst)[c] = c < live ? reinterpret_cast<const uint4*>(src)[c] : make_uint4(0, 0, 0, 0);
    return;
  }
  blk -= 8 * rows;
  const int chunk = blk % a.clear_chunks, item = blk / a.clear_chunks;
  const int bh = a.b0 * v.heads + item % rows, i = (item % rows) / v.heads, g = item / rows;
  Region r{};
#pragma unroll
  for (int k = 0; k < kRegions; ++k)
    if (k == g) r = a.region[k];
  const int used = r.kind == 0 ? a.len.packed[i] : (r.kind == 1 ? a.len.packed[i] / kGroup : a.len.late[r.kind - 2][i]);
  const int64_t from = static_cast<int64_t>(used) * r.unit + static_cast<int64_t>(chunk) * kClearBytes;
  const int64_t to = min(r.row, from + kClearBytes);
  uint8_t* p = r.base + bh * r.row;
  for (int64_t o = from + tid * 8; o < to; o += kBuildThreads * 8) *reinterpret_cast<uint2*>(p + o) = make_uint2(0, 0);
}

struct RollArgs {
  fl_cache_view v;
  int32_t* packed_tokens;
  int32_t* tail_tokens;
  int32_t* late_rows;
  uint8_t* tail_active[2];
  int32_t* scratch;  // [2, B]: destination group (-1: the sequence does not roll), tail rows left
};

// One wave per (b, s): a sequence whose tail holds a full group beyond the residual rows.
__global__ __launch_bounds__(kWave) void roll_begin_kernel(RollArgs a) {
  const fl_cache_view& v = a.v;
  const int b = blockIdx.x, s = blockIdx.y, lane = threadIdx.x;
  const int packed = a.packed_tokens[b], tail = a.tail_tokens[b];
  const bool roll = tail >= 2 * kGroup && packed >= 0 && packed % kGroup == 0 && packed + kGroup <= v.token_capacity;
  if (s == 0 && lane == 0) {
    a.scratch[b] = roll ? packed / kGroup : -1;
    a.scratch[v.batch + b] = min(tail, v.tail_capacity) - kGroup;
  }
  if (!roll) return;
  const bool on = a.tail_active[s][static_cast<int64_t>(b) * v.tail_capacity + lane] != 0;
  const uint64_t bits = __ballot(on);
  const int first = a.late_rows[s * v.batch + b];
  const int row = first + __popcll(bits & ((1ull << lane) - 1ull));
  v.rank[s][static_cast<int64_t>(b) * v.token_capacity + packed + lane] = on && row < v.row_capacity[2 + s] ? row : -1;
  if (lane == 0) a.late_rows[s * v.batch + b] = first + __popcll(bits);
}

// Workgroup (row bh, tensor): tail rows [64, 64 + n) to [0, n), 64 rows at a time in order, so a
// chunk is read before the next one's rows are written over it.  The y = 8 workgroups of each
// sequence's first head move its activity flags and set its lengths.
__global__ __launch_bounds__(kBuildThreads) void roll_end_kernel(RollArgs a) {
  const fl_cache_view& v = a.v;
  const int bh = blockIdx.x, t = blockIdx.y, b = bh / v.heads, tid = threadIdx.x;
  const int group = a.scratch[b];
  if (group < 0) return;
  const int n = a.scratch[v.batch + b];
  if (t == 8) {
    if (bh % v.heads != 0) return;
    for (int s = 0; s < 2; ++s) {
      uint8_t* act = (s == 0 ? a.tail_active[0] : a.tail_active[1]) + static_cast<int64_t>(b) * v.tail_capacity;
      for (int base = 0; base < v.tail_capacity; base += kGroup) {
        const int r = base + tid;
        const bool mine = tid < kGroup && r < v.tail_capacity;
        const uint8_t x = mine && r < n ? act[r + kGroup] : 0;
        __syncthreads();
        if (mine) act[r] = x;
      }
    }
    if (tid == 0) {
      a.packed_tokens[b] = (group + 1) * kGroup;
      a.tail_tokens[b] = n;
    }
    return;
  }
  uint16_t* p = nullptr;
#pragma unroll
  for (int k = 0; k < 8; ++k)
    if (k == t) p = k < 4 ? v.tail_key[k & 3] : v.tail_value[k & 3];
  p += static_cast<int64_t>(bh) * v.tail_capacity * kDim;
  constexpr int kChunk = kGroup * (kDim / 8);       // 16-byte pieces of 64 rows
  constexpr int kEach = kChunk / kBuildThreads;
  const int live = n * (kDim / 8);
  for (int base = 0; base < live; base += kChunk) {
    uint4 x[kEach];
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int c = base + tid + e * kBuildThreads;
      x[e] = c < live ? reinterpret_cast<const uint4*>(p)[c + kChunk] : make_uint4(0, 0, 0, 0);
    }
    __syncthreads();
#pragma unroll
    for (int e = 0; e < kEach; ++e) {
      const int c = base + tid + e * kBuildThreads;
      if (c < live) reinterpret_cast<uint4*>(p)[c] = x[e];
    }
  }
}
static_assert(kGroup * (kDim / 8) % kBuildThreads == 0, "whole pieces per thread");

}  // namespace
}  // namespace fl

extern "C" int32_t fl_count_active_rows(const uint8_t* const* masks, int64_t mask_stride, int32_t batch, int32_t tokens,
                                        const int32_t* packed, int32_t* counts, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(masks && packed && counts, "fl_count_active_rows: null argument");
  FL_REQUIRE(batch > 0 && tokens > 0 && mask_stride >= tokens, "fl_count_active_rows: bad sizes");
  for (int b = 0; b < batch; ++b)
    FL_REQUIRE(packed[b] >= 0 && packed[b] <= tokens, "fl_count_active_rows: a packed prefix exceeds the tokens");
  for (int b0 = 0; b0 < batch; b0 += kMaxSeqs) {
    const int seqs = std::min(kMaxSeqs, batch - b0);
    Lengths len{};
    for (int i = 0; i < seqs; ++i) len.packed[i] = packed[b0 + i];
    hipLaunchKernelGGL(count_active_kernel, dim3(seqs, 2), dim3(kBuildThreads), 0, static_cast<hipStream_t>(stream),
                       masks[0], masks[1], mask_stride, tokens, len, b0, batch, counts);
    FL_LAUNCH_CHECK("fl_count_active_rows");
  }
  return FL_OK;
}

extern "C" int32_t fl_cache_prepare(const fl_cache_view* view, const uint16_t* const* src_keys,
                                    const uint16_t* const* src_values, int64_t src_bh_stride,
                                    const uint8_t* const* masks, int64_t mask_stride, uint8_t* const* tail_active,
                                    const int32_t* packed, const int32_t* tail, const int32_t* late,
                                    int32_t* packed_tokens, int32_t* tail_tokens, int32_t* late_rows,
                                    int32_t* dst_group0, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(view && src_keys && src_values && masks && tail_active && packed && tail && late && packed_tokens &&
                 tail_tokens && late_rows && dst_group0, "fl_cache_prepare: null argument");
  const fl_cache_view& v = *view;
  FL_REQUIRE(v.batch > 0 && v.heads > 0 && v.tail_capacity > 0 && v.token_capacity > 0 && v.token_capacity % kGroup == 0,
             "fl_cache_prepare: bad view");
  PrepareArgs a{};
  a.v = v;
  a.src_stride = src_bh_stride;
  a.mask_stride = mask_stride;
  for (int r = 0; r < 4; ++r) {
    FL_REQUIRE(src_keys[r] && src_values[r] && v.tail_key[r] && v.tail_value[r] && v.key_codes[r] && v.key_meta[r] &&
                   v.value_meta[r] && v.key_meta_half[r] && v.value_meta_half[r],
               "fl_cache_prepare: null source or buffer");
    FL_REQUIRE(reinterpret_cast<uintptr_t>(src_keys[r]) % 16 == 0 && reinterpret_cast<uintptr_t>(src_values[r]) % 16 == 0,
               "fl_cache_prepare: sources must be 16-byte aligned");
    a.src[r] = src_keys[r];
    a.src[4 + r] = src_values[r];
  }
  FL_REQUIRE(v.value_meta_token && v.rank[0] && v.rank[1] && tail_active[0] && tail_active[1],
             "fl_cache_prepare: null buffer");
  for (int s = 0; s < 2; ++s) {
    a.mask[s] = masks[s];
    a.tail_active[s] = tail_active[s];
  }
  a.packed_tokens = packed_tokens;
  a.tail_tokens = tail_tokens;
  a.late_rows = late_rows;
  a.dst_group0 = dst_group0;
  const int cap = v.token_capacity, groups = cap / kGroup;
  int n = 0;
  const auto add = [&](void* base, int64_t units, int unit, int kind) {
    a.region[n++] = Region{static_cast<uint8_t*>(base), units * unit, unit, kind};
  };
  for (int s = 0; s < 4; ++s) {
    const int kind = s < 2 ? 0 : s;
    add(v.key_codes[s], v.row_capacity[s], kCodeStride, kind);
    add(v.key_meta[s], groups, kDim * 8, 1);
    add(v.value_meta[s], v.row_capacity[s], 16, kind);
    add(v.key_meta_half[s], groups, kDim * 4, 1);
    add(v.value_meta_half[s], v.row_capacity[s], 8, kind);
  }
  add(v.value_meta_token, cap, 64, 0);
  for (int b = 0; b < v.batch; ++b) {
    FL_REQUIRE(packed[b] >= 0 && packed[b] % kGroup == 0 && packed[b] <= cap && tail[b] >= 0 && tail[b] <= v.tail_capacity &&
                   static_cast<int64_t>(packed[b]) + tail[b] <= src_bh_stride,
               "fl_cache_prepare: lengths exceed the capacities or the sources");
    FL_REQUIRE((a.mask[0] == nullptr && a.mask[1] == nullptr) || static_cast<int64_t>(packed[b]) + tail[b] <= mask_stride,
               "fl_cache_prepare: mask_stride too small");
    for (int s = 0; s < 2; ++s)
      FL_REQUIRE(late[s * v.batch + b] >= 0 && late[s * v.batch + b] <= v.row_capacity[2 + s],
                 "fl_cache_prepare: late rows exceed the row capacity");
  }
  // workgroups of a launch over sequences b0 .. b0 + seqs - 1
  const auto plan = [&](int b0, int seqs) {
    int64_t unused = 0;  // the most bytes a (b,h) row of a region has to clear
    for (int i = 0; i < seqs; ++i)
      for (const Region& r : a.region) {
        const int used = r.kind == 0 ? packed[b0 + i]
                                     : (r.kind == 1 ? packed[b0 + i] / kGroup : late[(r.kind - 2) * v.batch + b0 + i]);
        unused = std::max(unused, r.row - static_cast<int64_t>(used) * r.unit);
      }
    const int64_t rows = static_cast<int64_t>(seqs) * v.heads;
    a.clear_chunks = static_cast<int>(std::max<int64_t>(1, (unused + kClearBytes - 1) / kClearBytes));
    return 3 * seqs + 8 * rows + (unused > 0 ? kRegions * rows * a.clear_chunks : 0);
  };
  constexpr int64_t kMaxBlocks = 0xFFFFFFFFll / kBuildThreads;  // 2^32 threads of a launch, past which it wraps
  for (int b0 = 0; b0 < v.batch; b0 += a.seqs) {
    a.b0 = b0;
    a.seqs = std::min(kMaxSeqs, v.batch - b0);
    int64_t blocks = plan(b0, a.seqs);
    while (blocks > kMaxBlocks && a.seqs > 1) {
      a.seqs = (a.seqs + 1) / 2;
      blocks = plan(b0, a.seqs);
    }
    FL_REQUIRE(blocks <= kMaxBlocks, "fl_cache_prepare: grid too large");
    for (int i = 0; i < a.seqs; ++i) {
      a.len.packed[i] = packed[b0 + i];
      a.len.tail[i] = tail[b0 + i];
      for (int s = 0; s < 2; ++s) a.len.late[s][i] = late[s * v.batch + b0 + i];
    }
    hipLaunchKernelGGL(cache_prepare_kernel, dim3(static_cast<unsigned>(blocks)), dim3(kBuildThreads), 0,
                       static_cast<hipStream_t>(stream), a);
    FL_LAUNCH_CHECK("fl_cache_prepare");
  }
  return FL_OK;
}

namespace {
int32_t roll_args(fl::RollArgs& a, const fl_cache_view* view, int32_t* packed_tokens, int32_t* tail_tokens,
                  int32_t* late_rows, uint8_t* const* tail_active, int32_t* scratch, const std::string& who) {
  using namespace fl;
  FL_REQUIRE(view && packed_tokens && tail_tokens && late_rows && tail_active && scratch, who + ": null argument");
  FL_REQUIRE(packed_tokens == view->packed_tokens && tail_tokens == view->tail_tokens,
             who + ": the lengths must be the view's arrays");
  FL_REQUIRE(view->batch > 0 && view->heads > 0 && view->tail_capacity >= 2 * kGroup && view->rank[0] && view->rank[1] &&
                 tail_active[0] && tail_active[1], who + ": bad view");
  for (int r = 0; r < 4; ++r) FL_REQUIRE(view->tail_key[r] && view->tail_value[r], who + ": null tail");
  a = RollArgs{*view, packed_tokens, tail_tokens, late_rows, {tail_active[0], tail_active[1]}, scratch};
  return FL_OK;
}
}  // namespace

extern "C" int32_t fl_roll_begin(const fl_cache_view* view, int32_t* packed_tokens, int32_t* tail_tokens,
                                 int32_t* late_rows, uint8_t* const* tail_active, int32_t* scratch, void* stream) {
  using namespace fl;
  clear_error();
  RollArgs a{};
  const int32_t rc = roll_args(a, view, packed_tokens, tail_tokens, late_rows, tail_active, scratch, "fl_roll_begin");
  if (rc != FL_OK) return rc;
  hipLaunchKernelGGL(roll_begin_kernel, dim3(view->batch, 2), dim3(kWave), 0, static_cast<hipStream_t>(stream), a);
  FL_LAUNCH_CHECK("fl_roll_begin");
  return FL_OK;
}

extern "C" int32_t fl_roll_end(const fl_cache_view* view, int32_t* packed_tokens, int32_t* tail_tokens,
                               int32_t* late_rows, uint8_t* const* tail_active, int32_t* scratch, void* stream) {
  using namespace fl;
  clear_error();
  RollArgs a{};
  const int32_t rc = roll_args(a, view, packed_tokens, tail_tokens, late_rows, tail_active, scratch, "fl_roll_end");
  if (rc != FL_OK) return rc;
  hipLaunchKernelGGL(roll_end_kernel, dim3(view->batch * view->heads, 9), dim3(kBuildThreads), 0,
                     static_cast<hipStream_t>(stream), a);
  FL_LAUNCH_CHECK("fl_roll_end");
  return FL_OK;
}
