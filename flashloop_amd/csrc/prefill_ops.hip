// Prefill row ops between the dense contractions of one sequence's prompt
// (flashloop/prefill.py:158-304), each one pass over its rows.
//
//  * fl_rope_store -- rotary embedding of the q and k rows that the projections wrote
//    ([n, heads * 128]), k and v going to their places in [heads, rows, 128] K/V (row
//    positions[i], or i): apply_rope, the transposes to head-major K/V and, in a token-sparse
//    loop, the scatter of the active rows.
//  * fl_swiglu -- bf16(silu(gate)) * up.
//
// Both are memory-bound: 16-byte accesses, one thread per 16 values (two rotary halves of 8).
// Every rounding to bf16 is where the torch modules round.  At 8192 rows of 16 heads the
// rotary pass takes 41 us (201 MB, 4.9 TB/s), where torch's products, concatenations, sums and
// copies took 282 us; SwiGLU of 5632 columns 43 us (277 MB, 6.4 TB/s; torch's two passes: 85 us).
#include "fl_common.h"

namespace fl {
namespace {

struct RopeStoreArgs {
  const uint16_t* src[3];  // q, k, v rows, row stride src_row
  int64_t src_row;
  uint16_t* q_out;         // row stride src_row (may be q itself)
  uint16_t* dst[2];        // k, v: [heads, rows, 128], head stride dst_head
  int64_t dst_head;
  const uint16_t* cos;     // [positions, 128] bf16
  const uint16_t* sin;
  const int32_t* positions;
  int n, heads, rows;
};

__device__ __forceinline__ void unpack_bf16x8(const uint4& u, float* f) {
  const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    f[2 * i] = bf16lo_to_f32(w[i]);
    f[2 * i + 1] = bf16hi_to_f32(w[i]);
  }
}

typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));
__device__ __forceinline__ uint32_t pack_bf16_pair(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}
__device__ __forceinline__ uint4 pack_bf16x8(const float* f) {
  return make_uint4(pack_bf16_pair(f[0], f[1]), pack_bf16_pair(f[2], f[3]), pack_bf16_pair(f[4], f[5]),
                    pack_bf16_pair(f[6], f[7]));
}
// eight values rounded to bf16 and widened again
__device__ __forceinline__ void round8(float* f) {
  const uint4 u = pack_bf16x8(f);
  unpack_bf16x8(u, f);
}

// Thread: 8 channels c..c+7 and their rotary partners c+64..c+71 of one row and head;
// blockIdx.y picks q, k or v.
__global__ __launch_bounds__(256) void rope_store_kernel(RopeStoreArgs a) {
  const int64_t t = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  const int64_t item = t >> 3;
  if (item >= static_cast<int64_t>(a.n) * a.heads) return;
  const int64_t i = item / a.heads;
  const int head = static_cast<int>(item - i * a.heads);
  const int c = static_cast<int>(t & 7) * 8;
  const int which = blockIdx.y;
  const int64_t row = a.positions ? a.positions[i] : i;
  if (row < 0 || row >= a.rows) return;
  const uint16_t* src = (which == 0 ? a.src[0] : (which == 1 ? a.src[1] : a.src[2])) + i * a.src_row + head * kDim + c;
  uint4 lo = *reinterpret_cast<const uint4*>(src);
  uint4 hi = *reinterpret_cast<const uint4*>(src + 64);
  if (which < 2) {
    const uint16_t* cs = a.cos + row * kDim + c;
    const uint16_t* sn = a.sin + row * kDim + c;
    float x[8], y[8], u[8], w[8], p[8], r[8];
    unpack_bf16x8(lo, x);
    unpack_bf16x8(hi, y);
    // lo' = bf16(bf16(x cos) + bf16(-y sin))
    unpack_bf16x8(*reinterpret_cast<const uint4*>(cs), u);
    unpack_bf16x8(*reinterpret_cast<const uint4*>(sn), w);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = x[e] * u[e];
      r[e] = -y[e] * w[e];
    }
    round8(p);
    round8(r);
#pragma unroll
    for (int e = 0; e < 8; ++e) p[e] += r[e];
    lo = pack_bf16x8(p);
    // hi' = bf16(bf16(y cos) + bf16(x sin))
    unpack_bf16x8(*reinterpret_cast<const uint4*>(cs + 64), u);
    unpack_bf16x8(*reinterpret_cast<const uint4*>(sn + 64), w);
#pragma unroll
    for (int e = 0; e < 8; ++e) {
      p[e] = y[e] * u[e];
      r[e] = x[e] * w[e];
    }
    round8(p);
    round8(r);
#pragma unroll
    for (int e = 0; e < 8; ++e) p[e] += r[e];
    hi = pack_bf16x8(p);
  }
  uint16_t* dst = which == 0 ? a.q_out + i * a.src_row + head * kDim + c
                             : (which == 1 ? a.dst[0] : a.dst[1]) + head * a.dst_head + row * kDim + c;
  *reinterpret_cast<uint4*>(dst) = lo;
  *reinterpret_cast<uint4*>(dst + 64) = hi;
}

__global__ __launch_bounds__(256) void swiglu_kernel(const uint16_t* gate, const uint16_t* up, uint16_t* out,
                                                     int64_t chunks) {
  const int64_t q = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (q >= chunks) return;
  float g[8], u[8];
  unpack_bf16x8(reinterpret_cast<const uint4*>(gate)[q], g);
  unpack_bf16x8(reinterpret_cast<const uint4*>(up)[q], u);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] = g[e] / (1.0f + expf(-g[e]));
  round8(g);
#pragma unroll
  for (int e = 0; e < 8; ++e) g[e] *= u[e];
  reinterpret_cast<uint4*>(out)[q] = pack_bf16x8(g);
}

bool aligned16(const void* p) { return reinterpret_cast<uintptr_t>(p) % 16 == 0; }

}  // namespace
}  // namespace fl

extern "C" int32_t fl_rope_store(const uint16_t* q, const uint16_t* k, const uint16_t* v, int64_t row_stride,
                                 uint16_t* q_out, uint16_t* k_dst, uint16_t* v_dst, int64_t dst_head_stride,
                                 const uint16_t* rope_cos, const uint16_t* rope_sin, const int32_t* positions,
                                 int32_t n, int32_t heads, int32_t rows, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(q && k && v && q_out && k_dst && v_dst && rope_cos && rope_sin, "fl_rope_store: null pointer");
  FL_REQUIRE(n >= 0 && heads > 0 && rows > 0, "fl_rope_store: bad sizes");
  FL_REQUIRE(positions != nullptr || n <= rows, "fl_rope_store: more rows than the destination without positions");
  FL_REQUIRE(row_stride >= static_cast<int64_t>(heads) * kDim && row_stride % 8 == 0 && dst_head_stride % 8 == 0,
             "fl_rope_store: bad strides");
  for (const void* p : {static_cast<const void*>(q), static_cast<const void*>(k), static_cast<const void*>(v),
                        static_cast<const void*>(q_out), static_cast<const void*>(k_dst),
                        static_cast<const void*>(v_dst), static_cast<const void*>(rope_cos),
                        static_cast<const void*>(rope_sin)})
    FL_REQUIRE(aligned16(p), "fl_rope_store: every tensor must be 16-byte aligned");
  if (n == 0) return FL_OK;
  const int64_t blocks = (static_cast<int64_t>(n) * heads * 8 + 255) / 256;
  FL_REQUIRE(blocks <= 0xFFFFFFFFll / 256, "fl_rope_store: grid too large");
  const RopeStoreArgs a{{q, k, v}, row_stride, q_out, {k_dst, v_dst}, dst_head_stride, rope_cos, rope_sin, positions,
                        n, heads, rows};
  hipLaunchKernelGGL(rope_store_kernel, dim3(static_cast<unsigned>(blocks), 3), dim3(256), 0,
                     static_cast<hipStream_t>(stream), a);
  FL_LAUNCH_CHECK("fl_rope_store");
  return FL_OK;
}

extern "C" int32_t fl_swiglu(const uint16_t* gate, const uint16_t* up, uint16_t* out, int64_t count, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(gate && up && out, "fl_swiglu: null pointer");
  FL_REQUIRE(count >= 0 && count % 8 == 0, "fl_swiglu: count must be a multiple of 8");
  FL_REQUIRE(aligned16(gate) && aligned16(up) && aligned16(out), "fl_swiglu: every tensor must be 16-byte aligned");
  if (count == 0) return FL_OK;
  const int64_t blocks = (count / 8 + 255) / 256;
  FL_REQUIRE(blocks <= 0xFFFFFFFFll / 256, "fl_swiglu: grid too large");
  hipLaunchKernelGGL(swiglu_kernel, dim3(static_cast<unsigned>(blocks)), dim3(256), 0, static_cast<hipStream_t>(stream),
                     gate, up, out, count / 8);
  FL_LAUNCH_CHECK("fl_swiglu");
  return FL_OK;
}
