// J4: token-sparse update row movement and the loop-boundary token score.
//
// fl_gather_rows / fl_scatter_rows move whole rows (hidden states, K/V rows) between a
// full tensor and its compact active-row copy: index_select / index_copy_ of
// flashloop/prefill.py:158, 193-194, 237 and flashloop/engine.py:276-333.  Every
// thread moves 16 bytes when rows and strides allow it, 4 bytes otherwise.
//
// fl_hidden_delta_score is _hidden_delta_score (flashloop/engine.py:78-81), one wave
// per row.
#include <algorithm>

#include "fl_common.h"

namespace fl {
namespace {

// Thread (item = one V of one moved row, outer): consecutive threads take the V's of a row and
// then of the next index, so short rows (a K/V row is 16 V's) still fill their waves -- with one
// workgroup per row 15/16 of the lanes idled: 2048 rows of 16 heads x 256 bytes 17 us, now 5.
// OWN: the flag is written (workgroup 0 looks at every index), not only set.
template <typename V, bool SCATTER, bool OWN>
__global__ __launch_bounds__(256) void move_rows_kernel(const uint8_t* src, int64_t s_outer, int64_t s_row,
                                                        uint8_t* dst, int64_t d_outer, int64_t d_row, int64_t rows,
                                                        uint32_t row_vecs, int64_t items, const int32_t* index,
                                                        int64_t n_index, int32_t* err) {
  if (OWN && blockIdx.x == 0 && blockIdx.y == 0) {
    __shared__ int bad;
    if (threadIdx.x == 0) bad = 0;
    __syncthreads();
    bool any = false;
    for (int64_t base = threadIdx.x; base < n_index; base += 8 * 256) {
      int32_t t[8];  // eight loads in flight (past the end: the last index again)
#pragma unroll
      for (int k = 0; k < 8; ++k) t[k] = index[base + k * 256 < n_index ? base + k * 256 : n_index - 1];
#pragma unroll
      for (int k = 0; k < 8; ++k) any |= t[k] < 0 || t[k] >= rows;
    }
    if (any) bad = 1;
    __syncthreads();
    if (threadIdx.x == 0) *err = bad;
  }
  const int64_t item = static_cast<int64_t>(blockIdx.x) * 256 + threadIdx.x;
  if (item >= items) return;
  const int64_t i = static_cast<uint32_t>(item) / row_vecs;
  const int64_t e = item - i * row_vecs;
  const int64_t o = blockIdx.y;
  const int32_t t = index[i];
  if (t < 0 || t >= rows) {
    if (!OWN && err && e == 0) atomicExch(err, 1);
    return;
  }
  const int64_t src_row = SCATTER ? i : t;
  const int64_t dst_row = SCATTER ? t : i;
  const V* s = reinterpret_cast<const V*>(src + o * s_outer + src_row * s_row) + e;
  V* d = reinterpret_cast<V*>(dst + o * d_outer + dst_row * d_row) + e;
  *d = *s;
}

template <bool SCATTER, bool OWN>
int32_t launch_move(const void* src, int64_t s_outer, int64_t s_row, void* dst, int64_t d_outer, int64_t d_row,
                    int64_t rows, int64_t outer, int64_t row_bytes, const int32_t* index, int64_t n_index,
                    int32_t* err, void* stream, const char* who) {
  FL_REQUIRE(src && dst && index, std::string(who) + ": null pointer");
  FL_REQUIRE(outer >= 0 && n_index >= 0 && rows >= 0 && row_bytes >= 0, std::string(who) + ": negative size");
  FL_REQUIRE(row_bytes % 4 == 0 && s_outer % 4 == 0 && s_row % 4 == 0 && d_outer % 4 == 0 && d_row % 4 == 0,
             std::string(who) + ": row bytes and strides must be multiples of 4");
  FL_REQUIRE(reinterpret_cast<uintptr_t>(src) % 4 == 0 && reinterpret_cast<uintptr_t>(dst) % 4 == 0,
             std::string(who) + ": pointers must be 4-byte aligned");
  FL_REQUIRE(n_index <= 65535 * 1024LL && outer <= 65535, std::string(who) + ": grid too large");
  const bool vec16 = row_bytes % 16 == 0 && s_outer % 16 == 0 && s_row % 16 == 0 && d_outer % 16 == 0 &&
                     d_row % 16 == 0 && reinterpret_cast<uintptr_t>(src) % 16 == 0 &&
                     reinterpret_cast<uintptr_t>(dst) % 16 == 0;
  const bool empty = outer == 0 || n_index == 0 || row_bytes == 0;
  if (empty && !OWN) return FL_OK;
  const int64_t vecs = empty ? 1 : (vec16 ? row_bytes / 16 : row_bytes / 4);
  constexpr int64_t kMaxItems = 0xFFFFFFFFll / 256 * 256;  // threads of a launch
  FL_REQUIRE(vecs <= kMaxItems, std::string(who) + ": rows too large");
  hipStream_t st = static_cast<hipStream_t>(stream);
  const uint8_t* s = static_cast<const uint8_t*>(src);
  uint8_t* d = static_cast<uint8_t*>(dst);
  // one launch up to 2^32 pieces of an outer index; of several, the first writes the flag for all
  const int64_t step = empty ? 1 : kMaxItems / vecs;
  int64_t i0 = 0;
  do {
    const int64_t items = empty ? 0 : vecs * std::min(step, n_index - i0);
    const dim3 grid(static_cast<unsigned>(std::max<int64_t>(1, (items + 255) / 256)), static_cast<unsigned>(empty ? 1 : outer));
    const auto go = [&](auto kernel, int32_t* flag) {
      hipLaunchKernelGGL(kernel, grid, dim3(256), 0, st, s + (SCATTER ? i0 * s_row : 0), s_outer, s_row,
                         d + (SCATTER ? 0 : i0 * d_row), d_outer, d_row, rows, static_cast<uint32_t>(vecs), items, index + i0,
                         n_index - i0, flag);
    };
    if (OWN && i0 > 0)
      vec16 ? go(move_rows_kernel<uint4, SCATTER, false>, nullptr) : go(move_rows_kernel<uint32_t, SCATTER, false>, nullptr);
    else
      vec16 ? go(move_rows_kernel<uint4, SCATTER, OWN>, err) : go(move_rows_kernel<uint32_t, SCATTER, OWN>, err);
    i0 += step;
  } while (!empty && i0 < n_index);
  FL_LAUNCH_CHECK(who);
  return FL_OK;
}

// One wave per row.  WIDE: 16-byte loads, four chunks of each row in flight per lane (rows of a
// multiple of 8 values, 16-byte aligned); 8192 rows of 2048: 17.4 us with 2-byte loads, 12.0.  From
// 256 values on, a chunk for half of the lanes: 32768 / 8192 / 100 rows of 512 take 16.3 / 3.8 / 2.8 us
// with 2-byte loads and 11.3 / 3.6 / 2.3 wide, of 256 9.2 / 3.3 / 2.4 and 8.6 / 3.5 / 2.3, of 128 6.5 / 3.1 /
// 2.2 and 8.1 / 3.6 / 2.4.
template <bool WIDE>
__global__ __launch_bounds__(256) void hidden_delta_score_kernel(const uint16_t* cur, const uint16_t* prev,
                                                                 int64_t rows, int dim, float* score) {
  const int64_t r = static_cast<int64_t>(blockIdx.x) * 4 + (threadIdx.x >> 6);
  if (r >= rows) return;
  const int lane = threadIdx.x & 63;
  const uint16_t* c = cur + r * dim;
  const uint16_t* p = prev + r * dim;
  float num = 0.0f, den = 0.0f;
  const auto add = [&](float a, float b) __attribute__((always_inline)) {
    const float d = a - b;
    num = fmaf(d, d, num);
    den = fmaf(a, a, den);
  };
  if constexpr (WIDE) {
    const int chunks = dim / 8;
    for (int q0 = lane; q0 < chunks; q0 += 4 * kWave) {
      uint4 x[4], y[4];
#pragma unroll
      for (int k = 0; k < 4; ++k) {  // (a chunk past the row repeats its last, and is not added)
        const int q = min(q0 + k * kWave, chunks - 1);
        x[k] = reinterpret_cast<const uint4*>(c)[q];
        y[k] = reinterpret_cast<const uint4*>(p)[q];
      }
#pragma unroll
      for (int k = 0; k < 4; ++k)
        if (q0 + k * kWave < chunks) {
          const uint32_t u[4] = {x[k].x, x[k].y, x[k].z, x[k].w}, v[4] = {y[k].x, y[k].y, y[k].z, y[k].w};
#pragma unroll
          for (int e = 0; e < 4; ++e) {
            add(bf16lo_to_f32(u[e]), bf16lo_to_f32(v[e]));
            add(bf16hi_to_f32(u[e]), bf16hi_to_f32(v[e]));
          }
        }
    }
  } else {
    for (int i = lane; i < dim; i += kWave) add(bf16_to_f32(c[i]), bf16_to_f32(p[i]));
  }
  num = wave_sum(num);
  den = wave_sum(den);
  if (lane == 0) score[r] = sqrtf(num) / fmaxf(sqrtf(den), 1e-12f);
}

}  // namespace
}  // namespace fl

extern "C" int32_t fl_gather_rows(const void* src, int64_t src_outer_stride, int64_t src_row_stride, int64_t src_rows,
                                  void* dst, int64_t dst_outer_stride, int64_t dst_row_stride, int64_t outer,
                                  int64_t row_bytes, const int32_t* index, int64_t n_index, int32_t* error_flag,
                                  void* stream) {
  fl::clear_error();
  return fl::launch_move<false, false>(src, src_outer_stride, src_row_stride, dst, dst_outer_stride, dst_row_stride,
                                src_rows, outer, row_bytes, index, n_index, error_flag, stream, "fl_gather_rows");
}

extern "C" int32_t fl_scatter_rows(const void* src, int64_t src_outer_stride, int64_t src_row_stride, void* dst,
                                   int64_t dst_outer_stride, int64_t dst_row_stride, int64_t dst_rows, int64_t outer,
                                   int64_t row_bytes, const int32_t* index, int64_t n_index, int32_t* error_flag,
                                   void* stream) {
  fl::clear_error();
  return fl::launch_move<true, false>(src, src_outer_stride, src_row_stride, dst, dst_outer_stride, dst_row_stride,
                               dst_rows, outer, row_bytes, index, n_index, error_flag, stream, "fl_scatter_rows");
}

extern "C" int32_t fl_move_rows(int32_t scatter, const void* src, int64_t src_outer_stride, int64_t src_row_stride,
                                void* dst, int64_t dst_outer_stride, int64_t dst_row_stride, int64_t indexed_rows,
                                int64_t outer, int64_t row_bytes, const int32_t* index, int64_t n_index,
                                int32_t* error_flag, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(error_flag != nullptr, "fl_move_rows: null error_flag");
  return scatter ? launch_move<true, true>(src, src_outer_stride, src_row_stride, dst, dst_outer_stride, dst_row_stride,
                                           indexed_rows, outer, row_bytes, index, n_index, error_flag, stream,
                                           "fl_move_rows")
                 : launch_move<false, true>(src, src_outer_stride, src_row_stride, dst, dst_outer_stride, dst_row_stride,
                                            indexed_rows, outer, row_bytes, index, n_index, error_flag, stream,
                                            "fl_move_rows");
}

extern "C" int32_t fl_hidden_delta_score(const uint16_t* cur, const uint16_t* prev, int64_t rows, int32_t dim,
                                         float* score, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(cur && prev && score, "fl_hidden_delta_score: null pointer");
  FL_REQUIRE(rows >= 0 && dim > 0, "fl_hidden_delta_score: bad shape");
  if (rows == 0) return FL_OK;
  const dim3 grid(static_cast<unsigned>((rows + 3) / 4));
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (dim % 8 == 0 && dim >= 4 * kWave && reinterpret_cast<uintptr_t>(cur) % 16 == 0 && reinterpret_cast<uintptr_t>(prev) % 16 == 0)
    hipLaunchKernelGGL(hidden_delta_score_kernel<true>, grid, dim3(256), 0, st, cur, prev, rows, dim, score);
  else
    hipLaunchKernelGGL(hidden_delta_score_kernel<false>, grid, dim3(256), 0, st, cur, prev, rows, dim, score);
  FL_LAUNCH_CHECK("fl_hidden_delta_score");
  return FL_OK;
}
