// Prefill attention: causal softmax(q K^T) V of one sequence's heads over bf16 rows, for a
// dense prompt (query i at position i) or for the active rows of a token-sparse loop (query
// i at positions[i]) -- the SDPA calls of flashloop/prefill.py:122-304.
//
// One workgroup of 4 waves owns 128 queries of one head, a wave 32 of them; the keys come in
// tiles of 64 through LDS, the next tile's global loads in flight while a tile is computed.
// Both contractions run on v_mfma_f32_32x32x16_bf16 with the queries as columns:
//   S^T[key, query] = K . Q^T      (A: K rows from LDS, B: the wave's Q, in registers)
//   O^T[d, query]  += V^T . P^T    (A: V columns, read transposed by ds_read_b64_tr_b16)
// so a lane holds one query throughout: its scores of a tile are 32 registers of two lanes,
// the softmax needs one lane exchange per tile, and P goes from the first product's result
// into the second's operand in place: result register r of lane half h is key
// 8 (r / 4) + 4 h + r % 4, and the second product takes its k in that order from V too.
// A tile rescales the accumulators only when some query's maximum grew (a wave vote): most do
// not.  (Raising the maximum only past 2^8 saves 4% more, but the largest probability is then
// no longer exactly 1 in bf16: error against 64 bits 2.05e-3 instead of 2.00e-3 at 2048 keys.)
//
// Bound by the matrix cores, the softmax's VALU work (quarter-rate exp) and the LDS reads at
// about the same rate each, so two workgroups share a CU (76 KB of LDS).  Measured, 16 heads, 8192
// dense queries: 338-370 us back to back (745-815 TFLOP/s of the causal half), 380 among the other
// kernels of a prompt (725); the SDPA it replaces: 725-740 us.  2048 of 8192: 118 us, 2000 937 -> 133;
// 820 of 8192: 940 -> 72 us.
#include <algorithm>
#include <cfloat>

#include "fl_common.h"

namespace fl {
namespace {

constexpr int kAttnWaves = 4;
constexpr int kAttnThreads = kAttnWaves * kWave;
constexpr int kQueries = 32 * kAttnWaves;  // per workgroup
constexpr int kKeys = 64;                  // per tile
// LDS rows: K padded by 16 bytes (the 16 lanes of a ds_read_b128 phase cover all banks), V
// by 64 (the four rows of a transposed 16-lane read lie 16 banks apart)
constexpr int kKRow = kDim + 8;
constexpr int kVRow = kDim + 32;

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef __bf16 bf16x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
typedef float f32x16_t __attribute__((ext_vector_type(16)));
typedef uint32_t u32x4_t __attribute__((ext_vector_type(4)));
typedef uint32_t u32x2_t __attribute__((ext_vector_type(2)));

struct AttnArgs {
  const uint16_t* q;  // query i of head h: q + h * q_head + i * q_row
  const uint16_t* k;
  const uint16_t* v;
  uint16_t* o;
  const int32_t* positions;  // [n], or null: query i is at position i
  int64_t q_head, q_row, k_head, k_row, v_head, v_row, o_head, o_row;
  int n, keys, heads;
  float scale;  // scaling * log2(e)
  int splits;   // key ranges per query block
  float* part_o;   // splits > 1: f32 [splits][n * heads][128], row i * heads + h
  float* part_ml;  // f32 [splits][n * heads][2]: maximum of q.k and sum
};

__device__ __forceinline__ uint32_t attn_bf16_pair(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}

// acc + both values of a packed bf16 pair (v_dot2_f32_bf16 with ones): the fp32 sum of the
// probabilities as the second product sees them, so that their roundings cancel in the quotient.
// The sum of the unrounded ones is 1-3% faster and errs more: against 64 bits 2.00e-3 instead of
// 1.99e-3 at 2048 dense queries, 2.03e-3 and 2.02e-3 at 8192 (the SDPA: 2.03e-3 and 2.08e-3).
__device__ __forceinline__ float add_pair(uint32_t w, float acc) {
  const bf16x2_t one = {static_cast<__bf16>(1.0f), static_cast<__bf16>(1.0f)};
  return __builtin_amdgcn_fdot2_f32_bf16(__builtin_bit_cast(bf16x2_t, w), one, acc, false);
}

// the other half-wave's value of the same query
__device__ __forceinline__ float swap_half(float v) { return __shfl_xor(v, 32, kWave); }

struct AttnLds {
  uint16_t k[2][kKeys * kKRow];
  uint16_t v[2][kKeys * kVRow];
};

// Base-2 logits past kFar: their products with the scale are no longer exact to a small part of 1, so
// that exp2(fma(s, scale, -m)) would be off by a power of two, or overflow.  There the differences
// are taken before the scale.  kNone: the maximum of a query that has seen no key.
constexpr float kFar = 4096.0f;
constexpr float kNone = -FLT_MAX;
__device__ __forceinline__ float scaled_max(float r, float scale) { return fmaxf(r * scale, -FLT_MAX); }
// 2^(scale (a - b)) of two raw maxima, a <= b; sa, sb: their scaled_max
__device__ __forceinline__ float exp2_between(float a, float b, float sa, float sb, float scale) {
  return fast_exp2(fabsf(sa) > kFar || fabsf(sb) > kFar ? (a - b) * scale : sa - sb);
}

// 4 keys (rows of the tile) of one d per lane: lane i of each 16-lane group passes the
// address of V[key + i / 4][d + 4 (i % 4)] and receives V[key .. key + 3][d + i].
__device__ __forceinline__ bf16x4_t read_v_tr(const uint16_t* p) {
  typedef __attribute__((address_space(3))) bf16x4_t lds_t;
  return __builtin_amdgcn_ds_read_tr16_b64_v4bf16(
      reinterpret_cast<lds_t*>(reinterpret_cast<uintptr_t>(p)));
}

template <bool SPLIT>
__global__ __launch_bounds__(kAttnThreads, 2) void attention_kernel(AttnArgs a) {
  __shared__ AttnLds L;
  __shared__ int last_pos[kAttnWaves];
  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6, h = lane >> 5;
  const int head = blockIdx.x % a.heads;
  const int blocks = (a.n + kQueries - 1) / kQueries;
  const int rest = static_cast<int>(blockIdx.x) / a.heads;
  const int split = SPLIT ? rest % a.splits : 0;
  const int qb = blocks - 1 - (SPLIT ? rest / a.splits : rest);  // longest key ranges first
  const int qi = qb * kQueries + wave * 32 + (lane & 31);
  const int qc = min(qi, a.n - 1);
  const int pos = a.positions ? a.positions[qc] : qc;
  int wmin = pos, wmax = pos;
#pragma unroll
  for (int off = 16; off >= 1; off >>= 1) {
    wmin = min(wmin, __shfl_xor(wmin, off, kWave));
    wmax = max(wmax, __shfl_xor(wmax, off, kWave));
  }
  if (lane == 0) last_pos[wave] = wmax;

  bf16x8_t q[8];
  {
    const uint16_t* qp = a.q + head * a.q_head + qc * a.q_row + 8 * h;
#pragma unroll
    for (int s = 0; s < 8; ++s) q[s] = *reinterpret_cast<const bf16x8_t*>(qp + 16 * s);
  }
  const uint16_t* kp = a.k + head * a.k_head;
  const uint16_t* vp = a.v + head * a.v_head;
  // this thread's four 16-byte chunks of a tile: rows tid / 16 + 16 i, chunk tid % 16
  const int lrow = tid >> 4, lcol = (tid & 15) * 8;
  u32x4_t kr[4], vr[4];
  const auto fetch = [&](int tile) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      const int64_t row = min(tile * kKeys + lrow + 16 * i, a.keys - 1);  // rows past the end: masked below
      kr[i] = *reinterpret_cast<const u32x4_t*>(kp + row * a.k_row + lcol);
      vr[i] = *reinterpret_cast<const u32x4_t*>(vp + row * a.v_row + lcol);
    }
  };
  const auto stage = [&](int buf) __attribute__((always_inline)) {
#pragma unroll
    for (int i = 0; i < 4; ++i) {
      *reinterpret_cast<u32x4_t*>(&L.k[buf][(lrow + 16 * i) * kKRow + lcol]) = kr[i];
      *reinterpret_cast<u32x4_t*>(&L.v[buf][(lrow + 16 * i) * kVRow + lcol]) = vr[i];
    }
  };
  int first = 0;
  if (!SPLIT) {  // the first tile's loads need no position
    fetch(0);
    stage(0);
  }
  lds_barrier();
  int end = 0;
#pragma unroll
  for (int w = 0; w < kAttnWaves; ++w) end = max(end, last_pos[w]);
  int tiles = min(end, a.keys - 1) / kKeys + 1;
  if (SPLIT) {
    first = static_cast<int>(static_cast<int64_t>(tiles) * split / a.splits);
    tiles = static_cast<int>(static_cast<int64_t>(tiles) * (split + 1) / a.splits);
    if (first < tiles) {
      fetch(first);
      stage(0);
    }
    lds_barrier();
  }

  f32x16_t o[4];
#pragma unroll
  for (int d = 0; d < 4; ++d)
#pragma unroll
    for (int r = 0; r < 16; ++r) o[d][r] = 0.0f;
  // running maximum (of q.k, and scaled to base 2) and this lane's part of the sum
  float raw = kNone, m = scaled_max(kNone, a.scale), l = 0.0f;
  bool far = false;  // (wave-uniform) some query's maximum lies past kFar

  for (int tile = first; tile < tiles; ++tile) {
    const int buf = (tile - first) & 1;
    fetch(min(tile + 1, tiles - 1));
    if (tile * kKeys <= wmax) {  // (wave-uniform) some query of the wave sees this tile
      f32x16_t s[2];
#pragma unroll
      for (int b = 0; b < 2; ++b) {
#pragma unroll
        for (int r = 0; r < 16; ++r) s[b][r] = 0.0f;
        const uint16_t* kl = &L.k[buf][(32 * b + (lane & 31)) * kKRow + 8 * h];
#pragma unroll
        for (int st = 0; st < 8; ++st)
          s[b] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(*reinterpret_cast<const bf16x8_t*>(kl + 16 * st), q[st], s[b], 0, 0, 0);
      }
      if (tile * kKeys + kKeys - 1 > wmin) {  // keys past a query's position
        const int lim = pos - tile * kKeys - 4 * h;
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r)
            if (32 * b + 8 * (r >> 2) + (r & 3) > lim) s[b][r] = -INFINITY;
      }
      float mx = s[0][0];
#pragma unroll
      for (int b = 0; b < 2; ++b)
#pragma unroll
        for (int r = 0; r < 16; ++r) mx = fmaxf(mx, s[b][r]);
      mx = fmaxf(mx, swap_half(mx));
      if (__builtin_amdgcn_ballot_w64(mx > raw) != 0ull) {
        const float top = fmaxf(raw, mx), mn = scaled_max(top, a.scale);
        const float alpha = exp2_between(raw, top, m, mn, a.scale);
        raw = top;
        m = mn;
        l *= alpha;
        far = __builtin_amdgcn_ballot_w64(fabsf(m) > kFar && raw > kNone) != 0ull;
#pragma unroll
        for (int d = 0; d < 4; ++d)
#pragma unroll
          for (int r = 0; r < 16; ++r) o[d][r] *= alpha;
      }
      float off = -m;
      if (far) {
#pragma unroll
        for (int b = 0; b < 2; ++b)
#pragma unroll
          for (int r = 0; r < 16; ++r) s[b][r] -= raw;
        off = 0.0f;
      }
      float sum[4] = {0.0f, 0.0f, 0.0f, 0.0f};
      bf16x8_t p[4];
#pragma unroll
      for (int t = 0; t < 4; ++t) {
        u32x4_t w;
#pragma unroll
        for (int i = 0; i < 4; ++i) {
          const int r = 8 * (t & 1) + 2 * i;
          const float p0 = fast_exp2(fmaf(s[t >> 1][r], a.scale, off));
          const float p1 = fast_exp2(fmaf(s[t >> 1][r + 1], a.scale, off));
          w[i] = attn_bf16_pair(p0, p1);
          sum[i] = add_pair(w[i], sum[i]);
        }
        p[t] = __builtin_bit_cast(bf16x8_t, w);
      }
      l += (sum[0] + sum[1]) + (sum[2] + sum[3]);
      const int i16 = lane & 15;
      const uint16_t* vl = &L.v[buf][(4 * h + (i16 >> 2)) * kVRow + ((lane >> 4) & 1) * 16 + 4 * (i16 & 3)];
#pragma unroll
      for (int t = 0; t < 4; ++t)
#pragma unroll
        for (int d = 0; d < 4; ++d) {
          const bf16x4_t lo = read_v_tr(vl + (16 * t) * kVRow + 32 * d);
          const bf16x4_t hi = read_v_tr(vl + (16 * t + 8) * kVRow + 32 * d);
          const bf16x8_t va = __builtin_shufflevector(lo, hi, 0, 1, 2, 3, 4, 5, 6, 7);
          o[d] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(va, p[t], o[d], 0, 0, 0);
        }
    }
    stage(buf ^ 1);  // (read by every wave before the barrier that ended the previous tile)
    lds_barrier();
  }

  l += swap_half(l);
  if (SPLIT) {
    if (qi < a.n) {
      const int64_t row = static_cast<int64_t>(split) * a.n * a.heads + static_cast<int64_t>(qi) * a.heads + head;
      float* op = a.part_o + row * kDim + 4 * h;
#pragma unroll
      for (int d = 0; d < 4; ++d)
#pragma unroll
        for (int g = 0; g < 4; ++g)
          *reinterpret_cast<float4*>(op + 32 * d + 8 * g) =
              make_float4(o[d][4 * g], o[d][4 * g + 1], o[d][4 * g + 2], o[d][4 * g + 3]);
      if (h == 0) *reinterpret_cast<float2*>(a.part_ml + 2 * row) = make_float2(raw, l);
    }
    return;
  }
  const float inv = 1.0f / l;
  if (qi < a.n) {
    uint16_t* op = a.o + head * a.o_head + qi * a.o_row + 4 * h;
#pragma unroll
    for (int d = 0; d < 4; ++d)
#pragma unroll
      for (int g = 0; g < 4; ++g) {
        u32x2_t w;
        w[0] = attn_bf16_pair(o[d][4 * g] * inv, o[d][4 * g + 1] * inv);
        w[1] = attn_bf16_pair(o[d][4 * g + 2] * inv, o[d][4 * g + 3] * inv);
        *reinterpret_cast<u32x2_t*>(op + 32 * d + 8 * g) = w;
      }
  }
}

// Merges the key ranges of a split launch: 32 lanes per (query, head) row, 4 channels each.
__global__ __launch_bounds__(256) void attention_merge_kernel(AttnArgs a) {
  const int64_t rows = static_cast<int64_t>(a.n) * a.heads;
  const int64_t row = static_cast<int64_t>(blockIdx.x) * 8 + (threadIdx.x >> 5);
  if (row >= rows) return;
  const int c = (threadIdx.x & 31) * 4;
  float M = kNone;
  for (int s = 0; s < a.splits; ++s) M = fmaxf(M, a.part_ml[2 * (s * rows + row)]);
  const float sm = scaled_max(M, a.scale);
  float l = 0.0f;
  float4 o = make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  for (int s = 0; s < a.splits; ++s) {
    const float2 ml = *reinterpret_cast<const float2*>(a.part_ml + 2 * (s * rows + row));
    const float4 p = *reinterpret_cast<const float4*>(a.part_o + (s * rows + row) * kDim + c);
    const float w = exp2_between(ml.x, M, scaled_max(ml.x, a.scale), sm, a.scale);
    l = fmaf(w, ml.y, l);
    o.x = fmaf(w, p.x, o.x);
    o.y = fmaf(w, p.y, o.y);
    o.z = fmaf(w, p.z, o.z);
    o.w = fmaf(w, p.w, o.w);
  }
  const float inv = 1.0f / l;
  u32x2_t w;
  w[0] = attn_bf16_pair(o.x * inv, o.y * inv);
  w[1] = attn_bf16_pair(o.z * inv, o.w * inv);
  const int64_t i = row / a.heads, h = row - i * a.heads;
  *reinterpret_cast<u32x2_t*>(a.o + h * a.o_head + i * a.o_row + c) = w;
}

// Key ranges per query block: 512 workgroups fill the chip (two per CU) and the later query
// blocks of a causal call are the longer ones, so a call of fewer than 640 blocks divides them,
// down to 448 keys a range.  16 heads, us with 1 / 2 / 3 / 4 / 6 / 8 ranges: 2048 queries of
// 8192 keys (256 blocks) 194 / 128 / 116 / 118 / 125 / 140, 820 of 8192 (112) 181 / 103 / 79 /
// 67 / 64 / 69, 3277 of 32768 (416) 816 / 609 / 592 / 588, 8192 of 8192 (1024) 378 / 367 / 378.
int attention_splits(int heads, int queries, int keys) {
  const int64_t groups = (static_cast<int64_t>(queries) + kQueries - 1) / kQueries * heads;
  const int64_t s = groups > 0 ? (640 + groups - 1) / groups : 1;
  return static_cast<int>(std::max<int64_t>(1, std::min<int64_t>(std::min<int64_t>(s, 16), keys / 448)));
}

size_t split_bytes(int heads, int queries) {
  return static_cast<size_t>(queries) * heads * (kDim + 2) * sizeof(float);
}

}  // namespace
}  // namespace fl

extern "C" size_t fl_prefill_attention_workspace(int32_t heads, int32_t queries, int32_t keys) {
  using namespace fl;
  if (heads <= 0 || queries <= 0 || keys <= 0) return 0;
  const int s = attention_splits(heads, queries, keys);
  return s > 1 ? s * split_bytes(heads, queries) : 0;
}

extern "C" int32_t fl_prefill_attention(const uint16_t* q, int64_t q_head_stride, int64_t q_row_stride,
                                        const uint16_t* k, int64_t k_head_stride, int64_t k_row_stride,
                                        const uint16_t* v, int64_t v_head_stride, int64_t v_row_stride,
                                        uint16_t* out, int64_t out_head_stride, int64_t out_row_stride,
                                        int32_t heads, int32_t queries, int32_t keys, const int32_t* positions,
                                        float scaling, void* workspace, size_t workspace_bytes, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(q && k && v && out, "fl_prefill_attention: null pointer");
  FL_REQUIRE(heads > 0 && queries >= 0 && keys > 0, "fl_prefill_attention: bad heads/queries/keys");
  FL_REQUIRE(positions != nullptr || queries <= keys, "fl_prefill_attention: more queries than keys without positions");
  FL_REQUIRE(scaling > 0.0f, "fl_prefill_attention: scaling must be positive");
  for (const int64_t s : {q_head_stride, q_row_stride, k_head_stride, k_row_stride, v_head_stride, v_row_stride,
                          out_head_stride, out_row_stride})
    FL_REQUIRE(s >= 0 && s % 8 == 0, "fl_prefill_attention: strides must be multiples of 8 elements");
  for (const void* p : {static_cast<const void*>(q), static_cast<const void*>(k), static_cast<const void*>(v),
                        static_cast<const void*>(out)})
    FL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "fl_prefill_attention: every tensor must be 16-byte aligned");
  if (queries == 0) return FL_OK;
  const int64_t blocks = (static_cast<int64_t>(queries) + kQueries - 1) / kQueries;
  FL_REQUIRE(blocks * heads <= 0xFFFFFFFFll / kAttnThreads, "fl_prefill_attention: grid too large");
  AttnArgs a{q, k, v, out, positions, q_head_stride, q_row_stride, k_head_stride, k_row_stride,
             v_head_stride, v_row_stride, out_head_stride, out_row_stride, queries, keys, heads,
             scaling * kLog2e, attention_splits(heads, queries, keys), nullptr, nullptr};
  // as many splits as the workspace holds (none without one)
  const size_t one = split_bytes(heads, queries);
  if (workspace == nullptr || reinterpret_cast<uintptr_t>(workspace) % 16 != 0) workspace_bytes = 0;
  a.splits = static_cast<int>(std::min<size_t>(a.splits, workspace_bytes / one));
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 block(kAttnThreads);
  if (a.splits <= 1) {
    hipLaunchKernelGGL(attention_kernel<false>, dim3(static_cast<unsigned>(blocks * heads)), block, 0, st, a);
    FL_LAUNCH_CHECK("fl_prefill_attention");
    return FL_OK;
  }
  const int64_t rows = static_cast<int64_t>(queries) * heads;
  a.part_o = static_cast<float*>(workspace);
  a.part_ml = a.part_o + a.splits * rows * kDim;
  hipLaunchKernelGGL(attention_kernel<true>, dim3(static_cast<unsigned>(blocks * heads * a.splits)), block, 0, st, a);
  FL_LAUNCH_CHECK("fl_prefill_attention");
  hipLaunchKernelGGL(attention_merge_kernel, dim3(static_cast<unsigned>((rows + 7) / 8)), dim3(256), 0, st, a);
  FL_LAUNCH_CHECK("fl_prefill_attention(merge)");
  return FL_OK;
}
