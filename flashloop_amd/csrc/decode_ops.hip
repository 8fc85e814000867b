// Decode-step model kernels: the per-layer work around the cache readers, fused so that
// one decode step of a layer and loop is eight launches instead of ~60 (the step of
// flashloop/engine.py:396-537 on an Ouro-shaped sandwich-norm layer).
//
//  * fl_gemv_bf16 -- y[m, n] = sum_k x[m, k] * W[n, k] for m < M <= 8 (nn.Linear weights,
//    bf16, row-major [N, K]); fp32 accumulation; epilogues: plain bf16 out, f32 out of the
//    bf16-rounded value (lm_head(...).float()), + bf16 addend, SwiGLU of a gate and an up
//    matrix, or rotary embedding of q/k (and a plain v) from three matrices at once.
//  * fl_norm_chain -- the residual/RMSNorm chain between two GEMVs of one row:
//    h = r + n_a(x); optionally h = n_f(h); z = n_b(h).
//
// Every rounding to bf16 happens where the torch modules round (Linear output, RMSNorm
// output, each binary op of rotate-half RoPE, SiLU, the SwiGLU product, residual adds).
//
// The GEMVs are memory-bound (bytes = N * K * 2 + M * K * 2); gemv_mfma_kernel runs K up to 8192
// (one and two rows: 4096), gemv_flat_kernel (VALU dots, one workgroup per 4 rows) one and two
// rows up to 8192, gemv_kernel (the same in a loop) the longer ones.
#include "fl_common.h"

namespace fl {
namespace {

constexpr int kGemvWaves = 4;
constexpr int kGemvThreads = kGemvWaves * kWave;
constexpr int kRows = 4;  // output rows per workgroup
constexpr int kMaxM = 8;

enum GemvEpi : int { kEpiPlain = 0, kEpiF32 = 1, kEpiAdd = 2, kEpiSwiGlu = 3, kEpiRope = 4 };

struct GemvArgs {
  const void* x;  // [M, K] bf16, or f32 (rounded to bf16 on load) when x_f32
  int64_t x_stride;
  int x_f32;
  int M, K, N;  // N: rows of each matrix
  const uint16_t* w[3];  // plain/add/f32: w[0]; swiglu: gate w[0], up w[1]; rope: q, k, v
  void* y[3];            // outputs [M, N] (row stride y_stride); rope: q, k, v
  int64_t y_stride;
  const uint16_t* addend;  // kEpiAdd: [M, N] bf16 (row stride addend_stride)
  int64_t addend_stride;
  const uint16_t* cos;  // kEpiRope: [M, 128] bf16 tables of each row's position
  const uint16_t* sin;
  int head_dim;
};

__device__ __forceinline__ float bf16_round(float v) { return round_bf16(v); }

__device__ __forceinline__ void unpack8(const uint4& u, float* f) {
  f[0] = bf16lo_to_f32(u.x);
  f[1] = bf16hi_to_f32(u.x);
  f[2] = bf16lo_to_f32(u.y);
  f[3] = bf16hi_to_f32(u.y);
  f[4] = bf16lo_to_f32(u.z);
  f[5] = bf16hi_to_f32(u.z);
  f[6] = bf16lo_to_f32(u.w);
  f[7] = bf16hi_to_f32(u.w);
}

// A raw buffer resource over `bytes` bytes at p (wave-uniform): loads past the end (or
// from a resource of size 0) return zero.  Word 3 is the gfx9 raw-buffer format.
using BufRes = __amdgpu_buffer_rsrc_t;
__device__ __forceinline__ BufRes buf_res(const void* p, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), 0, static_cast<int>(bytes), 0x00020000);
}
__device__ __forceinline__ uint4 buf_load16(BufRes r, uint32_t off) {
  return __builtin_bit_cast(uint4, __builtin_amdgcn_raw_buffer_load_b128(r, static_cast<int>(off), 0, 0));
}

// x chunk q (8 values) of row m, as the bf16 values the Linear sees
template <bool XF32>
__device__ __forceinline__ void load_x8(const GemvArgs& a, int m, int q, float* f) {
  if (XF32) {
    const float4* p = reinterpret_cast<const float4*>(static_cast<const float*>(a.x) + m * a.x_stride + 8 * q);
    const float4 u = p[0], v = p[1];
    f[0] = bf16_round(u.x);
    f[1] = bf16_round(u.y);
    f[2] = bf16_round(u.z);
    f[3] = bf16_round(u.w);
    f[4] = bf16_round(v.x);
    f[5] = bf16_round(v.y);
    f[6] = bf16_round(v.z);
    f[7] = bf16_round(v.w);
  } else {
    unpack8(*reinterpret_cast<const uint4*>(static_cast<const uint16_t*>(a.x) + m * a.x_stride + 8 * q), f);
  }
}

// Rows of workgroup g.  Plain: 4 consecutive rows of w[0].  SwiGLU: 2 consecutive rows,
// each of the gate and of the up matrix.  RoPE: matrix g / (N/4); within it the rotary
// pair rows {c, c+1, c+64, c+65} of one head, c even < 64.
template <int EPI>
__device__ __forceinline__ void block_rows(const GemvArgs& a, int g, const uint16_t** rp, int* mat, int* n0) {
  if (EPI == kEpiSwiGlu) {
    const int n = 2 * g;
    rp[0] = a.w[0] + static_cast<int64_t>(n) * a.K;
    rp[1] = a.w[0] + static_cast<int64_t>(n + 1) * a.K;
    rp[2] = a.w[1] + static_cast<int64_t>(n) * a.K;
    rp[3] = a.w[1] + static_cast<int64_t>(n + 1) * a.K;
    *mat = 0;
    *n0 = n;
  } else if (EPI == kEpiRope) {
    const int per = a.N / kRows;
    const int m = g / per, gi = g - m * per;
    const int half = a.head_dim / 2, pairs = half / 2;  // row groups per head
    const int head = gi / pairs, c = 2 * (gi - head * pairs);
    const int n = head * a.head_dim + c;
    const uint16_t* w = a.w[m];
    rp[0] = w + static_cast<int64_t>(n) * a.K;
    rp[1] = w + static_cast<int64_t>(n + 1) * a.K;
    rp[2] = w + static_cast<int64_t>(n + half) * a.K;
    rp[3] = w + static_cast<int64_t>(n + half + 1) * a.K;
    *mat = m;
    *n0 = n;
  } else {
    const int n = kRows * g;
#pragma unroll
    for (int r = 0; r < kRows; ++r) rp[r] = a.w[0] + static_cast<int64_t>(n + r) * a.K;
    *mat = 0;
    *n0 = n;
  }
}

// Cross-wave reduction of the partial dots and the epilogue (wave 0, lane m writes row m).
template <int MT, int EPI>
__device__ __forceinline__ void gemv_finish(const GemvArgs& a, float (*acc)[kRows], float (*red)[MT][kRows], int mat,
                                            int n0) {
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      const float s = wave_sum(acc[m][r]);
      if (lane == 0) red[wave][m][r] = s;
    }
  __syncthreads();
  if (wave != 0 || lane >= a.M) return;
  const int m = lane;
  float v[kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    float s = 0.0f;
#pragma unroll
    for (int w = 0; w < kGemvWaves; ++w) s += red[w][m < MT ? m : 0][r];
    v[r] = bf16_round(s);  // the Linear's bf16 output
  }
  const int64_t yo = static_cast<int64_t>(m) * a.y_stride + n0;
  if (EPI == kEpiF32) {
    float* y = static_cast<float*>(a.y[0]) + yo;
#pragma unroll
    for (int r = 0; r < kRows; ++r) y[r] = v[r];
  } else if (EPI == kEpiPlain || EPI == kEpiAdd) {
    uint16_t* y = static_cast<uint16_t*>(a.y[0]) + yo;
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      float o = v[r];
      if (EPI == kEpiAdd) o = o + bf16_to_f32(a.addend[static_cast<int64_t>(m) * a.addend_stride + n0 + r]);
      y[r] = f32_to_bf16_rne(o);
    }
  } else if (EPI == kEpiSwiGlu) {
    // silu(gate) rounds to bf16 (F.silu on bf16), then the product rounds
    uint16_t* y = static_cast<uint16_t*>(a.y[0]) + yo;
#pragma unroll
    for (int r = 0; r < 2; ++r) {
      const float g = v[r], u = v[2 + r];
      const float s = bf16_round(g / (1.0f + expf(-g)));
      y[r] = f32_to_bf16_rne(s * u);
    }
  } else {  // rope: rows (c, c+1) and (c+64, c+65); rotate_half(x)[c] = -x[c+64], [c+64] = x[c]
    uint16_t* y = static_cast<uint16_t*>(a.y[mat]) + yo;
    const int half = a.head_dim / 2;
    if (mat == 2) {
      y[0] = f32_to_bf16_rne(v[0]);
      y[1] = f32_to_bf16_rne(v[1]);
      y[half] = f32_to_bf16_rne(v[2]);
      y[half + 1] = f32_to_bf16_rne(v[3]);
    } else {
      const int c = (n0 % a.head_dim);
      const uint16_t* cs = a.cos + static_cast<int64_t>(m) * a.head_dim;
      const uint16_t* sn = a.sin + static_cast<int64_t>(m) * a.head_dim;
#pragma unroll
      for (int e = 0; e < 2; ++e) {
        const float lo = v[e], hi = v[2 + e];
        const float cl = bf16_to_f32(cs[c + e]), sl = bf16_to_f32(sn[c + e]);
        const float ch = bf16_to_f32(cs[c + half + e]), sh = bf16_to_f32(sn[c + half + e]);
        y[e] = f32_to_bf16_rne(bf16_round(lo * cl) + bf16_round(-hi * sl));
        y[half + e] = f32_to_bf16_rne(bf16_round(hi * ch) + bf16_round(lo * sh));
      }
    }
  }
}

template <int MT, int EPI, bool XF32>
__global__ __launch_bounds__(kGemvThreads) void gemv_kernel(GemvArgs a) {
  __shared__ float red[kGemvWaves][MT][kRows];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const uint16_t* rp[kRows];
  int mat, n0;
  block_rows<EPI>(a, blockIdx.x, rp, &mat, &n0);
  float acc[MT][kRows];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < kRows; ++r) acc[m][r] = 0.0f;
  const int nq = a.K / 8;  // 16-byte chunks per row
  // chunk q = j*256 + wave*64 + lane: each wave reads 1 KB contiguous per row and step
  constexpr int kStep = kGemvWaves * kWave;
  int q = wave * kWave + lane;
  // two steps per iteration keep 8 row loads in flight per lane
  for (; q + kStep < nq; q += 2 * kStep) {
    uint4 w0[kRows], w1[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) {
      w0[r] = reinterpret_cast<const uint4*>(rp[r])[q];
      w1[r] = reinterpret_cast<const uint4*>(rp[r])[q + kStep];
    }
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < a.M) {
        float x0[8], x1[8];
        load_x8<XF32>(a, m, q, x0);
        load_x8<XF32>(a, m, q + kStep, x1);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
          float f[8];
          unpack8(w0[r], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[m][r] = fmaf(x0[e], f[e], acc[m][r]);
          unpack8(w1[r], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[m][r] = fmaf(x1[e], f[e], acc[m][r]);
        }
      }
    }
  }
  if (q < nq) {
    uint4 w0[kRows];
#pragma unroll
    for (int r = 0; r < kRows; ++r) w0[r] = reinterpret_cast<const uint4*>(rp[r])[q];
#pragma unroll
    for (int m = 0; m < MT; ++m) {
      if (m < a.M) {
        float x0[8];
        load_x8<XF32>(a, m, q, x0);
#pragma unroll
        for (int r = 0; r < kRows; ++r) {
          float f[8];
          unpack8(w0[r], f);
#pragma unroll
          for (int e = 0; e < 8; ++e) acc[m][r] = fmaf(x0[e], f[e], acc[m][r]);
        }
      }
    }
  }
  gemv_finish<MT, EPI>(a, acc, red, mat, n0);
}

// The GEMV with every chunk a thread owns (S of them per row, K <= S * 2048) requested
// at once as bounds-checked buffer loads: chunks past K and rows past M read as zero, so
// no load sits under a branch (the compiler's wait after a branch join drains every
// outstanding load).  Same accumulation order as gemv_kernel.
template <int MT, int EPI, bool XF32, int S>
__global__ __launch_bounds__(kGemvThreads) void gemv_flat_kernel(GemvArgs a) {
  __shared__ float red[kGemvWaves][MT][kRows];
  const uint16_t* rp[kRows];
  int mat, n0;
  block_rows<EPI>(a, blockIdx.x, rp, &mat, &n0);
  constexpr int kStep = kGemvThreads;
  constexpr uint32_t kXb = XF32 ? 4u : 2u;  // bytes per x element
  const uint32_t q = threadIdx.x;
  uint4 wv[S][kRows];
#pragma unroll
  for (int r = 0; r < kRows; ++r) {
    const BufRes wr = buf_res(rp[r], static_cast<uint32_t>(a.K) * 2u);
#pragma unroll
    for (int s = 0; s < S; ++s) wv[s][r] = buf_load16(wr, 16u * (q + s * kStep));
  }
  uint4 xv[MT][S][XF32 ? 2 : 1];
#pragma unroll
  for (int m = 0; m < MT; ++m) {
    const bool live = m < a.M;
    const BufRes xr = buf_res(live ? static_cast<const char*>(a.x) + static_cast<int64_t>(m) * a.x_stride * kXb : nullptr,
                              live ? static_cast<uint32_t>(a.K) * kXb : 0u);
#pragma unroll
    for (int s = 0; s < S; ++s) {
      const uint32_t off = 8u * kXb * (q + s * kStep);
      xv[m][s][0] = buf_load16(xr, off);
      if (XF32) xv[m][s][XF32 ? 1 : 0] = buf_load16(xr, off + 16u);
    }
  }
  float acc[MT][kRows];
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int r = 0; r < kRows; ++r) acc[m][r] = 0.0f;
#pragma unroll
  for (int m = 0; m < MT; ++m)
#pragma unroll
    for (int s = 0; s < S; ++s) {
      float x[8];
      if (XF32) {
        const uint4 u = xv[m][s][0], v = xv[m][s][XF32 ? 1 : 0];
        const uint32_t w8[8] = {u.x, u.y, u.z, u.w, v.x, v.y, v.z, v.w};
#pragma unroll
        for (int e = 0; e < 8; ++e) x[e] = bf16_round(__uint_as_float(w8[e]));
      } else {
        unpack8(xv[m][s][0], x);
      }
#pragma unroll
      for (int r = 0; r < kRows; ++r) {
        float f[8];
        unpack8(wv[s][r], f);
#pragma unroll
        for (int e = 0; e < 8; ++e) acc[m][r] = fmaf(x[e], f[e], acc[m][r]);
      }
    }
  gemv_finish<MT, EPI>(a, acc, red, mat, n0);
}

// ---------------------------------------------------------------------------------
// Residual / RMSNorm chain of one row (one workgroup per row).  Thread t owns the
// 8-value chunks t, t + 256, ... of the row; every global load (x, r and the three
// weight rows) is issued before the first reduction, so the chain costs one memory
// round trip plus its block reductions.
// RMSNorm(x) = bf16(w * (x * rsqrt(mean(x^2) + eps))) in fp32, as the model's module.
constexpr int kNormThreads = 256;
constexpr int kNormChunks = 4;  // 8-value chunks per thread: D <= 8192

struct NormArgs {
  int D;
  float eps;
  const uint16_t* x;   // [M, D] or null (then h = r)
  const uint16_t* r;   // [M, D] residual / input
  const uint16_t* wa;  // norm of x
  const uint16_t* wf;  // optional norm of h (replaces h)
  const uint16_t* wb;  // optional norm of h -> z
  uint16_t* h_out;     // optional
  uint16_t* z_out;     // optional
  int64_t stride;      // row stride of every [M, D] tensor
};

constexpr int kNormWaves = kNormThreads / kWave;

// Block sums through two LDS buffers used in turn: reduction k writes buffer k & 1 and
// every wave reads it before it reaches the barrier of reduction k + 1, so buffer k & 1 is
// free again for reduction k + 2 -- one barrier per sum.  Waves past the first kNormWaves
// of a larger workgroup take part in the barriers only.
struct BlockSum {
  float (*red)[kNormWaves];
  int phase;
  __device__ __forceinline__ float operator()(float v) {
    float* r = red[phase & 1];
    ++phase;
    v = wave_sum(v);
    if ((threadIdx.x & 63) == 0 && threadIdx.x < kNormThreads) r[threadIdx.x >> 6] = v;
    lds_barrier();  // (a global fence would wait for a caller's weight loads)
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < kNormWaves; ++i) s += r[i];
    return s;
  }
};

// v <- RMSNorm(v) with weight chunks w (8 values per chunk), rounded to bf16
template <int NC>
__device__ __forceinline__ void rms_apply(float (*v)[8], const uint4* w, int nc, int D, float eps, BlockSum& bs) {
  float ss = 0.0f;
#pragma unroll
  for (int i = 0; i < NC; ++i)
    if (i < nc)
#pragma unroll
      for (int e = 0; e < 8; ++e) ss = fmaf(v[i][e], v[i][e], ss);
  const float inv = rsqrtf(bs(ss) / static_cast<float>(D) + eps);
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    float wf[8];
    unpack8(w[i], wf);
#pragma unroll
    for (int e = 0; e < 8; ++e) v[i][e] = bf16_round(wf[e] * (v[i][e] * inv));
  }
}

__device__ __forceinline__ uint4 pack8(const float* f) {
  uint4 u;
  u.x = static_cast<uint32_t>(f32_to_bf16_rne(f[0])) | (static_cast<uint32_t>(f32_to_bf16_rne(f[1])) << 16);
  u.y = static_cast<uint32_t>(f32_to_bf16_rne(f[2])) | (static_cast<uint32_t>(f32_to_bf16_rne(f[3])) << 16);
  u.z = static_cast<uint32_t>(f32_to_bf16_rne(f[4])) | (static_cast<uint32_t>(f32_to_bf16_rne(f[5])) << 16);
  u.w = static_cast<uint32_t>(f32_to_bf16_rne(f[6])) | (static_cast<uint32_t>(f32_to_bf16_rne(f[7])) << 16);
  return u;
}

// The chain of row `base` (element offset): h = r (+ n_a(x)), optionally h = n_f(h),
// written to h_out when write_h; then z = n_b(h) when n_b is given.  chain_load issues the
// loads of this thread's chunks t, t + 256, ...; chain_finish leaves z (or h without n_b)
// in v as bf16 values.  All kNormThreads threads must call chain_finish (block reductions).
template <int NC>
struct ChainIn {
  uint4 xr[NC], rr[NC], wa[NC], wf[NC], wb[NC];
};

template <int NC>
__device__ __forceinline__ void chain_load(const NormArgs& a, int64_t base, ChainIn<NC>& in) {
  const int nq = a.D / 8;
  const int nc = (nq - static_cast<int>(threadIdx.x) + kNormThreads - 1) / kNormThreads;  // my chunks
  // Buffer loads sized to each operand (size 0 when absent): chunks past the row read as
  // zero without a branch.  A load under a branch would make the compiler's wait at the
  // join drain every outstanding load, including a caller's loads issued after these.
  (void)nc;
  const uint32_t row = static_cast<uint32_t>(a.D) * 2u;
  const BufRes r = buf_res(a.r + base, row);
  const BufRes x = buf_res(a.x ? a.x + base : nullptr, a.x ? row : 0u);
  const BufRes wa = buf_res(a.x ? a.wa : nullptr, a.x ? row : 0u);
  const BufRes wf = buf_res(a.wf, a.wf ? row : 0u);
  const BufRes wb = buf_res(a.wb, a.wb ? row : 0u);
#pragma unroll
  for (int i = 0; i < NC; ++i) {
    const uint32_t off = 16u * static_cast<uint32_t>(threadIdx.x + i * kNormThreads);
    in.rr[i] = buf_load16(r, off);
    in.xr[i] = buf_load16(x, off);
    in.wa[i] = buf_load16(wa, off);
    in.wf[i] = buf_load16(wf, off);
    in.wb[i] = buf_load16(wb, off);
  }
}

template <int NC>
__device__ __forceinline__ void chain_finish(const NormArgs& a, int64_t base, bool write_h, const ChainIn<NC>& in,
                                             float (*h)[8], BlockSum& bs) {
  const int nc = (a.D / 8 - static_cast<int>(threadIdx.x) + kNormThreads - 1) / kNormThreads;
#pragma unroll
  for (int i = 0; i < NC; ++i) unpack8(in.rr[i], h[i]);
  if (a.x != nullptr) {
    float xv[NC][8];
#pragma unroll
    for (int i = 0; i < NC; ++i) unpack8(in.xr[i], xv[i]);
    rms_apply<NC>(xv, in.wa, nc, a.D, a.eps, bs);
#pragma unroll
    for (int i = 0; i < NC; ++i)
#pragma unroll
      for (int e = 0; e < 8; ++e) h[i][e] = bf16_round(h[i][e] + xv[i][e]);
  }
  if (a.wf != nullptr) rms_apply<NC>(h, in.wf, nc, a.D, a.eps, bs);
  if (write_h && a.h_out != nullptr) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if (i < nc) reinterpret_cast<uint4*>(a.h_out + base)[threadIdx.x + i * kNormThreads] = pack8(h[i]);
  }
  if (a.wb != nullptr) rms_apply<NC>(h, in.wb, nc, a.D, a.eps, bs);
}

template <int NC>
__device__ __forceinline__ void chain_row(const NormArgs& a, int64_t base, bool write_h, float (*h)[8], BlockSum& bs) {
  ChainIn<NC> in;
  chain_load<NC>(a, base, in);
  chain_finish<NC>(a, base, write_h, in, h, bs);
}

template <int NC>
__global__ __launch_bounds__(kNormThreads) void norm_chain_kernel(NormArgs a) {
  __shared__ float red[2][kNormWaves];
  BlockSum bs{red, 0};
  const int64_t base = static_cast<int64_t>(blockIdx.x) * a.stride;
  const int nc = (a.D / 8 - static_cast<int>(threadIdx.x) + kNormThreads - 1) / kNormThreads;
  float h[NC][8];
  chain_row<NC>(a, base, true, h, bs);
  if (a.wb != nullptr) {
#pragma unroll
    for (int i = 0; i < NC; ++i)
      if (i < nc) reinterpret_cast<uint4*>(a.z_out + base)[threadIdx.x + i * kNormThreads] = pack8(h[i]);
  }
}

// ---------------------------------------------------------------------------------
// The GEMV of a decode step on the matrix cores, with the chain of its input rows in the
// prologue where there is one (bit-identical to norm_chain_kernel then this kernel: same
// chunk ownership, same order of the sums).
//
// v_mfma_f32_16x16x32_bf16 takes 16 rows of W and 16 columns of x over 32 k.  A decode step
// has 1 to 8 rows of x, so a tile is T rows of W by T rows of x (T = 8, or 4 for one row) and
// the rest of the instruction's rows and columns holds further k of the same rows: row i and
// column j are (row i % T, k-slice i / T) and (x row j % T, k-slice j / T).  The diagonal
// T x T blocks of the product add up to the tile (the others mix slices and are not used), and
// the lanes of one W row read 128 (T = 8) or 256 (T = 4) contiguous bytes per load.
//
// Bound by HBM and, for small matrices, by the launch's ramp: the VALU form it replaces cost
// M * K fused multiply-adds per W row, M sequential chains per workgroup and one chain per 4
// rows.  A unit of NT tiles (SwiGLU: gate and up rows; RoPE: rotary pairs) is one workgroup's
// work, all its weights requested before its first product; its waves split K in steps of 512
// and their partial tiles meet in LDS.  Eight rows take 8 waves, one wave per chain row; one
// row takes 4 waves and 4-row tiles (twice the workgroups).  Measured, 2048 wide (q/k/v with
// RoPE, o_proj, SwiGLU 5632, down, lm_head 49152), us before -> now: 8 rows 46.8 -> 10.0,
// 12.1 -> 5.4, 75.2 -> 12.9, 15.6 -> 7.9, 287 -> 40 (5.0 TB/s); one row 9.2 -> 7.7, 4.8 -> 4.9,
// 13.3 -> 10.8, down stays on the VALU form (6.1, 6.9 here), 42.0 -> 36.5 (5.5 TB/s).  One row with
// 8 waves and 8-row tiles took 9.1, 5.1, 11.9, 6.9 and 38.4.
template <int MT>
struct MmGeom {
  static constexpr int kWaves = MT == 1 ? 4 : 8;
  static constexpr int kThreads = kWaves * kWave;
  static constexpr int kTile = MT == 1 ? 4 : 8;    // rows of W (and of x) per tile
  static constexpr int kSlices = 16 / kTile;       // k-slices of 32 side by side in one MFMA
  static constexpr int kWaveK = 32 * kSlices;      // k of one MFMA
  static constexpr int kParts = kWaves * kSlices;  // partial tiles of a unit
};
constexpr int kMmStepK = 512;    // k of one step of all waves
constexpr int kChainMaxK = 4096;
constexpr int kMmMaxK = 8192;    // of the largest instantiation

typedef __bf16 bf16x8_t __attribute__((ext_vector_type(8)));
typedef float f32x4_t __attribute__((ext_vector_type(4)));
typedef __bf16 bf16x2_t __attribute__((ext_vector_type(2)));
typedef float f32x2_t __attribute__((ext_vector_type(2)));

// Two values rounded to bf16 and packed (v_cvt_pk_bf16_f32, nearest even, NaN kept NaN).
__device__ __forceinline__ uint32_t bf16_pair(float lo, float hi) {
  const f32x2_t f = {lo, hi};
  return __builtin_bit_cast(uint32_t, __builtin_convertvector(f, bf16x2_t));
}
__device__ __forceinline__ uint4 bf16_pack8(const float* f) {
  return make_uint4(bf16_pair(f[0], f[1]), bf16_pair(f[2], f[3]), bf16_pair(f[4], f[5]), bf16_pair(f[6], f[7]));
}

// Where a lane's tile rows of unit u lie: a buffer over the unit's rows and this lane's
// byte offset in it, per tile.  Rows past the matrix repeat its last row (not stored).
template <int NT>
struct UnitRows {
  BufRes res[NT];
  uint32_t off[NT];
};

__device__ __forceinline__ BufRes rows_res(const uint16_t* w, int64_t row, int64_t rows, int K) {
  const int64_t left = (rows - row) * K * 2;
  return buf_res(w + row * K, static_cast<uint32_t>(left < 0x7FFFFFFF ? left : 0x7FFFFFFF));
}

template <int EPI, int MT>
__host__ __device__ __forceinline__ int units_per_matrix(int n) {
  constexpr int kTile = MmGeom<MT>::kTile;
  return EPI == kEpiRope ? (n / 2 + kTile - 1) / kTile : (n + kTile - 1) / kTile;
}

// First k of this lane (its k-slice of its wave's MFMA).
template <int MT>
__device__ __forceinline__ int lane_k0() {
  using G = MmGeom<MT>;
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  return wave * G::kWaveK + ((lane & 15) / G::kTile) * 32 + (lane >> 4) * 8;
}

template <int EPI, int MT, int NT>
__device__ __forceinline__ void unit_rows(const GemvArgs& a, int u, UnitRows<NT>& ur) {
  constexpr int kTile = MmGeom<MT>::kTile;
  const int i = threadIdx.x & (kTile - 1);
  const uint32_t row_bytes = static_cast<uint32_t>(a.K) * 2u;
  if (EPI == kEpiSwiGlu) {
    const int n = kTile * u;
    const uint32_t row = static_cast<uint32_t>(min(i, a.N - 1 - n));
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      ur.res[t] = rows_res(a.w[t], n, a.N, a.K);
      ur.off[t] = row * row_bytes;
    }
  } else if (EPI == kEpiRope) {
    const int per = units_per_matrix<EPI, MT>(a.N), half = a.head_dim / 2;
    const int mat = u / per, p0 = (u - mat * per) * kTile;
    const int p = min(p0 + i, a.N / 2 - 1);
    const int n0 = (p0 / half) * a.head_dim + p0 % half;  // the unit's first row
    const int n = (p / half) * a.head_dim + p % half;
    const uint16_t* w = mat == 0 ? a.w[0] : (mat == 1 ? a.w[1] : a.w[2]);
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      ur.res[t] = rows_res(w, n0, a.N, a.K);
      ur.off[t] = static_cast<uint32_t>(n - n0 + t * half) * row_bytes;
    }
  } else {
    const int n = NT * kTile * u;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      ur.res[t] = rows_res(a.w[0], n, a.N, a.K);
      ur.off[t] = static_cast<uint32_t>(min(kTile * t + i, a.N - 1 - n)) * row_bytes;
    }
  }
}

// This wave's k of the unit's tiles: step s covers kWaveK values from s * 512 + wave * kWaveK;
// chunks past K lie outside the buffer and read as zero.
template <int MT, int NT, int CS>
__device__ __forceinline__ void load_unit(const UnitRows<NT>& ur, int K, uint4 (&w)[NT][CS]) {
  const int k0 = lane_k0<MT>();
#pragma unroll
  for (int s = 0; s < CS; ++s) {
    const int k = k0 + s * kMmStepK;
    const uint32_t ko = k < K ? 2u * static_cast<uint32_t>(k) : 0x80000000u;
#pragma unroll
    for (int t = 0; t < NT; ++t) w[t][s] = buf_load16(ur.res[t], ur.off[t] + ko);
  }
}

// What the epilogue of unit u reads besides the dots: cos and sin of the rotary pair, or the
// addends.  Requested right behind the unit's weights, so that no load follows the last product
// (8 rows: o_proj 5.7 -> 5.4 us; q/k/v with RoPE 11.3 -> 10.7).
template <int EPI, int NT>
struct EpiIn {
  uint16_t v[EPI == kEpiRope ? 4 : NT];
};

template <int EPI, int MT, int NT>
__device__ __forceinline__ void load_epi(const GemvArgs& a, int u, EpiIn<EPI, NT>& e) {
  constexpr int kTile = MmGeom<MT>::kTile;
  const int m = threadIdx.x / kTile, i = threadIdx.x % kTile;
  if (EPI == kEpiRope) {
    const int per = units_per_matrix<EPI, MT>(a.N), half = a.head_dim / 2;
    const int mat = u / per, p = (u - mat * per) * kTile + i;
    if (mat == 2 || m >= min(MT, a.M) || p >= a.N / 2) return;
    const int64_t o = static_cast<int64_t>(m) * a.head_dim + p % half;
    e.v[0] = a.cos[o];
    e.v[1] = a.sin[o];
    e.v[2] = a.cos[o + half];
    e.v[3] = a.sin[o + half];
  } else if (EPI == kEpiAdd) {
    if (m >= min(MT, a.M)) return;
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = (NT * u + t) * kTile + i;
      if (n < a.N) e.v[t] = a.addend[static_cast<int64_t>(m) * a.addend_stride + n];
    }
  }
}

// Output (m, i-th row of each tile) of unit u from the tiles' bf16-rounded dots v[t].
template <int EPI, int MT, int NT>
__device__ __forceinline__ void unit_store(const GemvArgs& a, int u, int m, int i, const float* v,
                                           const EpiIn<EPI, NT>& e) {
  constexpr int kTile = MmGeom<MT>::kTile;
  if (EPI == kEpiSwiGlu) {
    const int n = kTile * u + i;
    if (n >= a.N) return;
    const float g = v[0], up = v[NT - 1];
    const float s = bf16_round(g / (1.0f + expf(-g)));  // F.silu on bf16 rounds, then the product
    static_cast<uint16_t*>(a.y[0])[static_cast<int64_t>(m) * a.y_stride + n] = f32_to_bf16_rne(s * up);
  } else if (EPI == kEpiRope) {  // rotate_half(x)[c] = -x[c + half], [c + half] = x[c]
    const int per = units_per_matrix<EPI, MT>(a.N), half = a.head_dim / 2;
    const int mat = u / per, p = (u - mat * per) * kTile + i;
    if (p >= a.N / 2) return;
    const int c = p % half;
    const float lo = v[0], hi = v[NT - 1];
    uint16_t* y = static_cast<uint16_t*>(mat == 0 ? a.y[0] : (mat == 1 ? a.y[1] : a.y[2])) +
                  static_cast<int64_t>(m) * a.y_stride + (p / half) * a.head_dim + c;
    if (mat == 2) {
      y[0] = f32_to_bf16_rne(lo);
      y[half] = f32_to_bf16_rne(hi);
    } else {
      y[0] = f32_to_bf16_rne(bf16_round(lo * bf16_to_f32(e.v[0])) + bf16_round(-hi * bf16_to_f32(e.v[1])));
      y[half] = f32_to_bf16_rne(bf16_round(hi * bf16_to_f32(e.v[2])) + bf16_round(lo * bf16_to_f32(e.v[3])));
    }
  } else {
#pragma unroll
    for (int t = 0; t < NT; ++t) {
      const int n = (NT * u + t) * kTile + i;
      if (n >= a.N) return;
      const int64_t o = static_cast<int64_t>(m) * a.y_stride + n;
      if (EPI == kEpiF32)
        static_cast<float*>(a.y[0])[o] = v[t];
      else if (EPI == kEpiAdd)
        static_cast<uint16_t*>(a.y[0])[o] =
            f32_to_bf16_rne(v[t] + bf16_to_f32(e.v[t]));
      else
        static_cast<uint16_t*>(a.y[0])[o] = f32_to_bf16_rne(v[t]);
    }
  }
}

// One row's chain by one wave: lane l holds chunks l + 64 j, and the four partial sums of
// a norm are those of norm_chain_kernel's four waves (thread 64 w + l: chunks 64 w + l and
// 256 + 64 w + l), added in its order.
template <int CH>
struct WaveChainIn {
  uint4 x[CH], r[CH], wa[CH], wb[CH];
};

template <int CH>
__device__ __forceinline__ void wave_chain_load(const NormArgs& c, int64_t base, WaveChainIn<CH>& in) {
  const uint32_t row = static_cast<uint32_t>(c.D) * 2u;
  const BufRes r = buf_res(c.r + base, row);
  const BufRes x = buf_res(c.x ? c.x + base : nullptr, c.x ? row : 0u);
  const BufRes wa = buf_res(c.x ? c.wa : nullptr, c.x ? row : 0u);
  const BufRes wb = buf_res(c.wb, c.wb ? row : 0u);
  const uint32_t o = 16u * (threadIdx.x & 63u);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    in.x[j] = buf_load16(x, o + 1024u * j);
    in.r[j] = buf_load16(r, o + 1024u * j);
    in.wa[j] = buf_load16(wa, o + 1024u * j);
    in.wb[j] = buf_load16(wb, o + 1024u * j);
  }
}

template <int CH>
__device__ __forceinline__ void wave_rms(uint4 (&v)[CH], const uint4 (&w)[CH], int D, float eps) {
  float ss[4] = {0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    float f[8];
    unpack8(v[j], f);
#pragma unroll
    for (int e = 0; e < 8; ++e) ss[j & 3] = fmaf(f[e], f[e], ss[j & 3]);
  }
#pragma unroll
  for (int i = 0; i < 4; ++i) ss[i] = wave_sum(ss[i]);
  const float inv = rsqrtf((((ss[0] + ss[1]) + ss[2]) + ss[3]) / static_cast<float>(D) + eps);
#pragma unroll
  for (int j = 0; j < CH; ++j) {
    float f[8], g[8];
    unpack8(v[j], f);
    unpack8(w[j], g);
#pragma unroll
    for (int e = 0; e < 8; ++e) f[e] = g[e] * (f[e] * inv);
    v[j] = bf16_pack8(f);
  }
}

// z (or h without n_b) of the row, as packed bf16, in in.r; h is written to h_out when asked
template <int CH>
__device__ __forceinline__ void wave_chain(const NormArgs& c, int64_t base, bool write_h, WaveChainIn<CH>& in) {
  if (c.x != nullptr) {
    wave_rms<CH>(in.x, in.wa, c.D, c.eps);
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      float f[8], g[8];
      unpack8(in.r[j], f);
      unpack8(in.x[j], g);
#pragma unroll
      for (int e = 0; e < 8; ++e) f[e] += g[e];
      in.r[j] = bf16_pack8(f);
    }
  }
  if (c.wf != nullptr) {  // the last chain of a loop only: loaded here, so that the others keep the registers
    const BufRes res = buf_res(c.wf, static_cast<uint32_t>(c.D) * 2u);
#pragma unroll
    for (int j = 0; j < CH; ++j) in.x[j] = buf_load16(res, 16u * (threadIdx.x & 63u) + 1024u * j);
    wave_rms<CH>(in.r, in.x, c.D, c.eps);
  }
  if (write_h && c.h_out != nullptr) {
#pragma unroll
    for (int j = 0; j < CH; ++j) {
      const int q = static_cast<int>(threadIdx.x & 63u) + 64 * j;
      if (q < c.D / 8) reinterpret_cast<uint4*>(c.h_out + base)[q] = in.r[j];
    }
  }
  if (c.wb != nullptr) wave_rms<CH>(in.r, in.wb, c.D, c.eps);
}

// This lane's x chunks (k as in load_unit) of row lane % 8, rounded to bf16 when x is f32;
// zero past K (the weights there read as zero too) and in rows past M.
template <int MT, int CS>
__device__ __forceinline__ void load_x(const GemvArgs& a, bf16x8_t (&x)[CS]) {
  const int k0 = lane_k0<MT>();
  const int m = MT == 1 ? 0 : (threadIdx.x & 7);
  const uint32_t es = a.x_f32 ? 4u : 2u;
  const BufRes r = buf_res(a.x, (static_cast<uint32_t>(a.M - 1) * static_cast<uint32_t>(a.x_stride) + a.K) * es);
  const uint32_t row = static_cast<uint32_t>(m) * static_cast<uint32_t>(a.x_stride) * es;
  if (a.x_f32) {
    uint4 lo[CS], hi[CS];
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      const int k = k0 + s * kMmStepK;
      const uint32_t o = k < a.K && m < a.M ? row + 4u * static_cast<uint32_t>(k) : 0x80000000u;
      lo[s] = buf_load16(r, o);
      hi[s] = buf_load16(r, o + 16u);
    }
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      const float f[8] = {__uint_as_float(lo[s].x), __uint_as_float(lo[s].y), __uint_as_float(lo[s].z),
                          __uint_as_float(lo[s].w), __uint_as_float(hi[s].x), __uint_as_float(hi[s].y),
                          __uint_as_float(hi[s].z), __uint_as_float(hi[s].w)};
      x[s] = __builtin_bit_cast(bf16x8_t, bf16_pack8(f));
    }
  } else {
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      const int k = k0 + s * kMmStepK;
      const uint32_t o = k < a.K && m < a.M ? row + 2u * static_cast<uint32_t>(k) : 0x80000000u;
      x[s] = __builtin_bit_cast(bf16x8_t, buf_load16(r, o));
    }
  }
}

// KCAP: the largest K of the instantiation (a unit's weights are in registers).  MT: x rows
// (1, or up to 8).  DEPTH: units whose weights are in flight (1: a grid of one unit per workgroup;
// 2: of several).
template <int EPI, int MT, int KCAP, int NT, bool CHAIN, int DEPTH>
__global__ __launch_bounds__(MmGeom<MT>::kThreads, 2) void gemv_mfma_kernel(GemvArgs a, NormArgs c, int units) {
  using G = MmGeom<MT>;
  constexpr int CS = KCAP / kMmStepK;  // steps of a wave over K
  constexpr int kRow = KCAP + 8;       // x row in LDS, elements
  // one row with RoPE: three short workgroups a CU hide the load, its arithmetic up front costs 0.25 us
  constexpr bool kAhead = EPI == kEpiAdd || (EPI == kEpiRope && MT > 1);
  __shared__ uint16_t xs[CHAIN ? MT * kRow : 8];
  __shared__ float red[2][G::kParts][NT][MT][G::kTile];  // [unit parity][wave, k-slice][tile][x row][W row]
  __shared__ float nred[2][kNormWaves];
  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);  // (buffer descriptors of a wave's row are scalar)

  uint4 w[DEPTH][NT][CS];
  EpiIn<EPI, NT> e[DEPTH];
  int u = blockIdx.x;
  const int step = gridDim.x;
  const auto load = [&](int unit, int d) __attribute__((always_inline)) {
    UnitRows<NT> ur;
    const int K = DEPTH == 1 || unit < units ? a.K : 0;  // (past the last unit: nothing is read)
    if (DEPTH > 1) unit = min(unit, units - 1);
    unit_rows<EPI, MT, NT>(a, unit, ur);
    load_unit<MT, NT, CS>(ur, K, w[d]);
    // the weights are all requested here (left to itself the compiler loads each before its product
    // once no loop follows: K 5632 6.9 -> 7.4 us), and ahead of load_epi's index arithmetic
    __builtin_amdgcn_sched_barrier(0);
    if (kAhead && wave == 0) load_epi<EPI, MT, NT>(a, unit, e[d]);  // (the threads that store lie in one wave)
  };
  static_assert(MT * G::kTile <= kWave, "one wave stores");
  const auto load_first = [&]() __attribute__((always_inline)) {
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) load(u + d * step, d);
  };
  bf16x8_t xr[CHAIN ? 1 : CS];
  if constexpr (CHAIN && MT == 1) {
    // one row: the workgroup holds it as norm_chain_kernel does
    static_assert(G::kThreads == kNormThreads, "one GEMV thread per chain thread");
    constexpr int NC = KCAP / (kNormThreads * 8);
    ChainIn<NC> in;
    float z[NC][8];
    BlockSum bs{nred, 0};
    chain_load<NC>(c, 0, in);
    __builtin_amdgcn_sched_barrier(0);  // the chain's inputs return before the weights
    load_first();
    __builtin_amdgcn_sched_barrier(0);
    chain_finish<NC>(c, 0, blockIdx.x == 0, in, z, bs);
#pragma unroll
    for (int i = 0; i < NC; ++i)
      *reinterpret_cast<uint4*>(&xs[8 * (tid + i * kNormThreads)]) = bf16_pack8(z[i]);  // (zero past K)
  } else if constexpr (CHAIN) {
    constexpr int CH = KCAP / 512;
    WaveChainIn<CH> in;  // wave w: row w (rows past M repeat the last: columns no output reads)
    const int64_t base = static_cast<int64_t>(min(wave, a.M - 1)) * c.stride;
    wave_chain_load<CH>(c, base, in);
    __builtin_amdgcn_sched_barrier(0);
    load_first();
    __builtin_amdgcn_sched_barrier(0);
    if (wave < a.M) {
      wave_chain<CH>(c, base, blockIdx.x == 0, in);
#pragma unroll
      for (int j = 0; j < CH; ++j) *reinterpret_cast<uint4*>(&xs[wave * kRow + 8 * (lane + 64 * j)]) = in.r[j];
    }
  } else {
    load_x<MT, CS>(a, xr);
    load_first();
  }
  if constexpr (CHAIN) lds_barrier();

  const uint16_t* xl = &xs[CHAIN ? (MT == 1 ? 0 : (lane & 7)) * kRow + lane_k0<MT>() : 0];
  int par = 0;
  const auto compute = [&](int d, int unit) __attribute__((always_inline)) {
    f32x4_t acc[NT];
#pragma unroll
    for (int t = 0; t < NT; ++t) acc[t] = f32x4_t{0.0f, 0.0f, 0.0f, 0.0f};
#pragma unroll
    for (int s = 0; s < CS; ++s) {
      bf16x8_t xv;
      if constexpr (CHAIN)
        xv = *reinterpret_cast<const bf16x8_t*>(xl + s * kMmStepK);
      else
        xv = xr[s];
#pragma unroll
      for (int t = 0; t < NT; ++t)
        acc[t] = __builtin_amdgcn_mfma_f32_16x16x32_bf16(__builtin_bit_cast(bf16x8_t, w[d][t][s]), xv, acc[t], 0, 0, 0);
    }
    // lane l holds rows 4 (l / 16) ..+3 of column l % 16: the diagonal blocks are kept
    const int row = 4 * (lane >> 4), col = lane & 15;
    if (row / G::kTile == col / G::kTile && col % G::kTile < MT)
#pragma unroll
      for (int t = 0; t < NT; ++t)
        *reinterpret_cast<f32x4_t*>(&red[par][wave * G::kSlices + row / G::kTile][t][col % G::kTile][row % G::kTile]) = acc[t];
    lds_barrier();
    if (tid < MT * G::kTile) {
      const int m = tid / G::kTile, i = tid % G::kTile;
      if (m < a.M) {
        float v[NT];
#pragma unroll
        for (int t = 0; t < NT; ++t) {
          float sum = 0.0f;
#pragma unroll
          for (int p = 0; p < G::kParts; ++p) sum += red[par][p][t][m][i];
          v[t] = bf16_round(sum);  // the Linear's bf16 output
        }
        if constexpr (!kAhead) load_epi<EPI, MT, NT>(a, unit, e[d]);
        unit_store<EPI, MT, NT>(a, unit, m, i, v, e[d]);
      }
    }
    par ^= 1;  // (a buffer is written again after the next unit's barrier)
  };
  for (;; u += DEPTH * step)
#pragma unroll
    for (int d = 0; d < DEPTH; ++d) {
      compute(d, u + d * step);
      if (DEPTH == 1 || u + (d + 1) * step >= units) return;
      load(u + (d + DEPTH) * step, d);
    }
}

// ---------------------------------------------------------------------------------
// Decode append: the step's K/V rows of the four loops go to each sequence's tail at its
// device length, the loop-3/4 activity flags of that row are set, and the length is
// incremented -- one workgroup per sequence and layer, so the increment follows its own copies.
// Bound by its launch, so a step's layers share one (a step of four layers 923 -> 916 us).
constexpr int kAppendThreads = 256;
constexpr int kAppendLayers = 16;  // per launch (kernel arguments: 160 bytes a layer)

struct AppendLayer {
  uint16_t* tail[8];       // tail_key of the four loops, then tail_value
  const uint16_t* rows[8];  // [B*H, 128] bf16 rows of the step: keys, then values
  uint8_t* active[2];      // [B, tail_capacity] loop-3/4 tail activity
  int32_t* tail_tokens;    // the tail lengths, written
};
struct AppendArgs {
  int heads, tail_capacity;
  AppendLayer layer[kAppendLayers];
};

__global__ __launch_bounds__(kAppendThreads) void append_tail_kernel(AppendArgs a) {
  const AppendLayer& l = a.layer[blockIdx.y];
  const int b = blockIdx.x;
  constexpr int kChunks = kDim / 8;     // 16-byte chunks per row
  const int per = a.heads * kChunks;    // chunks of one tensor for this sequence
  auto src_of = [&](int t, int i) __attribute__((always_inline)) {
    return reinterpret_cast<const uint4*>(l.rows[t] + static_cast<int64_t>(b) * a.heads * kDim) + i;
  };
  auto dst_of = [&](int t, int i, int pos) __attribute__((always_inline)) {
    const int h = i / kChunks, c = i - h * kChunks;
    return reinterpret_cast<uint4*>(l.tail[t] + ((static_cast<int64_t>(b) * a.heads + h) * a.tail_capacity + pos) * kDim) + c;
  };
  // chunk threadIdx.x of each of the 8 tensors is requested before the first store (the
  // rows do not depend on the tail length, loaded alongside): one memory round trip
  const int pos = l.tail_tokens[b];
  const int i0 = threadIdx.x;
  uint4 held[8];
#pragma unroll
  for (int t = 0; t < 8; ++t) held[t] = i0 < per ? *src_of(t, i0) : make_uint4(0, 0, 0, 0);
  if (pos < 0 || pos >= a.tail_capacity) return;  // the host rolls over before the tail is full
#pragma unroll
  for (int t = 0; t < 8; ++t)
    if (i0 < per) *dst_of(t, i0, pos) = held[t];
  for (int i = i0 + kAppendThreads; i < per; i += kAppendThreads)  // more than 16 heads
#pragma unroll
    for (int t = 0; t < 8; ++t) *dst_of(t, i, pos) = *src_of(t, i);
  if (threadIdx.x < 2) l.active[threadIdx.x][static_cast<int64_t>(b) * a.tail_capacity + pos] = 1;
  __syncthreads();
  if (threadIdx.x == 0) l.tail_tokens[b] = pos + 1;
}

// ---------------------------------------------------------------------------------
// Inputs of a decode step: the token's embedding row and the cos / sin rows of its position, one
// workgroup per sequence.  One dependent load and one chain of conversions, so it is bound by its
// launch: with it in place of the seven launches of the two modules (and the logits written where
// the caller reads them) a four-layer step takes 923 us, 941 before.
constexpr int kInputThreads = 256;

struct InputArgs {
  const int64_t* tokens;     // [B]
  const int64_t* positions;  // [B]
  const uint16_t* table;     // [vocab, D]
  int64_t vocab;
  int D, half;               // half: head_dim / 2
  const void* inv_freq;      // [half] f32 or bf16
  int freq_bf16;
  uint16_t* h;               // [B, D]
  uint16_t* cos;             // [B, 2 * half]
  uint16_t* sin;
};

__global__ __launch_bounds__(kInputThreads) void decode_inputs_kernel(InputArgs a) {
  const int b = blockIdx.x, tid = threadIdx.x;
  const int64_t tok = a.tokens[b];
  const float pos = static_cast<float>(a.positions[b]);
  const bool in = tok >= 0 && tok < a.vocab;  // (a token outside the table gives NaN, never a read)
  const uint4* row = reinterpret_cast<const uint4*>(a.table + (in ? tok : 0) * a.D);
  uint4* h = reinterpret_cast<uint4*>(a.h + static_cast<int64_t>(b) * a.D);
  for (int c = tid; c < a.D / 8; c += kInputThreads)
    h[c] = in ? row[c] : make_uint4(0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u, 0x7FC07FC0u);
  for (int i = tid; i < a.half; i += kInputThreads) {
    const float f = a.freq_bf16 ? bf16_to_f32(static_cast<const uint16_t*>(a.inv_freq)[i])
                                : static_cast<const float*>(a.inv_freq)[i];
    const float angle = pos * f;
    const int64_t o = static_cast<int64_t>(b) * 2 * a.half + i;
    a.cos[o] = a.cos[o + a.half] = f32_to_bf16_rne(cosf(angle));
    a.sin[o] = a.sin[o + a.half] = f32_to_bf16_rne(sinf(angle));
  }
}

template <int EPI, int MT, int KCAP, int NT, bool CHAIN, int DEPTH>
void launch_gemv_mfma(const GemvArgs& a, const NormArgs& c, int workgroups, hipStream_t st) {
  const int per = units_per_matrix<EPI, MT>(a.N);
  const int units = EPI == kEpiRope ? 3 * per : (EPI == kEpiSwiGlu ? per : (per + NT - 1) / NT);
  int grid = units;
  if (DEPTH > 1) {  // at most `workgroups`, each with the same number of units
    const int rounds = (units + workgroups - 1) / workgroups;
    grid = (units + rounds - 1) / rounds;
  }
  hipLaunchKernelGGL((gemv_mfma_kernel<EPI, MT, KCAP, NT, CHAIN, DEPTH>), dim3(grid), dim3(MmGeom<MT>::kThreads), 0, st, a, c, units);
}

// The forms give a row the same products in the same order, so a chained call and its GEMV apart
// may take different ones.  Each reads K in steps of 512 up to its KCAP, so one is there for every
// 1024 or 2048 of K: one row without a chain, K 1024, lm_head 49152 and SwiGLU 5632 22.1 and 7.3 us
// on the 2048 form, 18.1 and 6.5 on their own; K 3072 56.2 and 15.8 on the 4096 form, 46.5 and 14.1.
//
// Several units per workgroup (DEPTH 2) where the prologue or the epilogue of one unit would not
// hide behind the other workgroups of its CU.  Eight chained rows: the prologue is ~700 VALU
// instructions per row, so one workgroup per CU runs it once (SwiGLU 5632 x 2048: 16.8 us with
// a workgroup per unit, 12.9 with 235 of three units; three units in flight gain nothing there
// and q/k/v with RoPE, two units each, loses 9.9 -> 10.6).  One chained row: only the many units of
// a head-sized matrix gain (lm_head 49152 x 2048: 37.5 -> 36.3 us, x 3072 67.8 -> 54.2, x 4096 79.4
// -> 69.9; SwiGLU lost, 10.8 -> 13.1).  Without a chain one or two rows lose by it (lm_head 49152 x
// 2048 31.3 -> 35.7 and 33.9 -> 36.5 us), three rows and more gain (eight 47.5 -> 38.5).
//
// Two tiles a unit where the workgroups are many: a short K of a head-sized matrix (eight rows,
// lm_head 49152 x 1024 24.9 -> 21.5 us), and f32 rows, whose x loads cost as much as a tile's
// weights (4096 x 4096 with an addend, one row 9.7 -> 8.6, eight 13.9 -> 11.3; not below one
// workgroup a CU: two rows, 2048 x 4096 6.1 -> 7.2).
template <int EPI, int MT, bool CHAIN>
void launch_gemv_k(const GemvArgs& a, const NormArgs& c, hipStream_t st) {
  constexpr int kPair = EPI == kEpiSwiGlu || EPI == kEpiRope ? 2 : 1;
  const bool head = kPair == 1 && a.N >= 16384;
  if constexpr (CHAIN) {
    if (a.K <= 2048) {
      if constexpr (MT == 8) {
        launch_gemv_mfma<EPI, MT, 2048, 2, true, 2>(a, c, 256, st);
      } else {
        if (a.N >= 16384) return launch_gemv_mfma<EPI, MT, 2048, 2, true, 2>(a, c, 1024, st);
        launch_gemv_mfma<EPI, MT, 2048, kPair, true, 1>(a, c, 0, st);
      }
    } else {
      if constexpr (MT == 1 && kPair == 1)
        if (head) return launch_gemv_mfma<EPI, MT, 4096, 1, true, 2>(a, c, 1024, st);
      launch_gemv_mfma<EPI, MT, 4096, kPair, true, 1>(a, c, 0, st);
    }
  } else if (a.K <= 1024) {
    if constexpr (kPair == 1)
      if (head) return launch_gemv_mfma<EPI, MT, 1024, 2, false, 1>(a, c, 0, st);
    launch_gemv_mfma<EPI, MT, 1024, kPair, false, 1>(a, c, 0, st);
  } else if (a.K <= 2048) {
    if constexpr (MT == 8)
      if (a.N >= 16384 && (kPair == 2 || a.M > 2)) return launch_gemv_mfma<EPI, MT, 2048, 2, false, 2>(a, c, 1024, st);
    launch_gemv_mfma<EPI, MT, 2048, kPair, false, 1>(a, c, 0, st);
  } else if (a.K <= 3072) {
    launch_gemv_mfma<EPI, MT, 3072, kPair, false, 1>(a, c, 0, st);
  } else if (a.K <= 4096) {
    if constexpr (kPair == 1)
      if (a.x_f32 && a.N >= 256 * 2 * MmGeom<MT>::kTile)
        return launch_gemv_mfma<EPI, MT, 4096, 2, false, 1>(a, c, 0, st);
    launch_gemv_mfma<EPI, MT, 4096, kPair, false, 1>(a, c, 0, st);
  } else if constexpr (MT > 1) {
    if (a.K <= 6144)
      launch_gemv_mfma<EPI, MT, 6144, kPair, false, 1>(a, c, 0, st);
    else
      launch_gemv_mfma<EPI, MT, kMmMaxK, kPair, false, 1>(a, c, 0, st);
  }
}

// Workgroups of the kernels of one workgroup per kRows rows.
template <int EPI>
int gemv_blocks(int n) {
  return EPI == kEpiSwiGlu ? n / 2 : (EPI == kEpiRope ? 3 * (n / kRows) : n / kRows);
}

template <int EPI, bool XF32>
void launch_gemv_long(const GemvArgs& a, hipStream_t st) {
  const dim3 g(gemv_blocks<EPI>(a.N)), t(kGemvThreads);
  // (no more rows of accumulators than the call has: two rows, K 10240 to 2048, on the eight-row form
  // 12.4 -> 14.4 us, four rows 15.7 -> 17.0)
  if (a.M <= 1)
    hipLaunchKernelGGL((gemv_kernel<1, EPI, XF32>), g, t, 0, st, a);
  else if (a.M <= 2)
    hipLaunchKernelGGL((gemv_kernel<2, EPI, XF32>), g, t, 0, st, a);
  else if (a.M <= 4)
    hipLaunchKernelGGL((gemv_kernel<4, EPI, XF32>), g, t, 0, st, a);
  else
    hipLaunchKernelGGL((gemv_kernel<8, EPI, XF32>), g, t, 0, st, a);
}

// One and two rows of K 4104 to 8192: the matrix cores' 16 k-slices of partial sums and x loads per
// unit cost more than the rows' own VALU dots.  To 2048, us with them and without: one row K 5632
// 6.9 -> 6.1, 8192 9.0 -> 8.0, two rows 7.1 -> 6.8 and 9.3 -> 8.6, SwiGLU 5632 x 8192 34.4 -> 31.3
// and 37.5 -> 31.4; from three rows on they lose (K 5632 8.8 against 7.3).  Up to 4096 one and two
// rows stay on the matrix cores too, with the bits of the chained call: q/k/v with RoPE and SwiGLU
// of 2048 are 7.2 and 10.2 us there against 7.0 and 9.8 (the chained call 7.4 and 10.9 against 8.7
// and 13.1).
template <int MT, int EPI, bool XF32>
void launch_gemv_flat(const GemvArgs& a, hipStream_t st) {
  const dim3 g(gemv_blocks<EPI>(a.N)), t(kGemvThreads);
  if (a.K <= 6144)
    hipLaunchKernelGGL((gemv_flat_kernel<MT, EPI, XF32, 3>), g, t, 0, st, a);
  else
    hipLaunchKernelGGL((gemv_flat_kernel<MT, EPI, XF32, 4>), g, t, 0, st, a);
}

// K up to 8192 (a unit's weights in registers) runs on the matrix cores, one and two rows up to
// 4096, further on gemv_flat_kernel; longer rows, and heads or x strides so wide that a unit's rows
// do not fit one buffer, on gemv_kernel.
template <int EPI, bool CHAIN>
void launch_gemv(const GemvArgs& a, const NormArgs& c, hipStream_t st) {
  if constexpr (!CHAIN)
    if (a.M <= 2 && a.K > kChainMaxK && a.K <= kMmMaxK) {
      if (a.M == 1) return a.x_f32 ? launch_gemv_flat<1, EPI, true>(a, st) : launch_gemv_flat<1, EPI, false>(a, st);
      return a.x_f32 ? launch_gemv_flat<2, EPI, true>(a, st) : launch_gemv_flat<2, EPI, false>(a, st);
    }
  const bool wide = (EPI == kEpiRope && (static_cast<int64_t>(a.head_dim) + 16) * a.K * 2 > 0x7FFFFFFF) ||
                    (a.M > 1 && a.x_stride > 0x7FFFFFFF / (4 * kMaxM));
  if (CHAIN || (a.K <= kMmMaxK && !wide)) {
    if (a.M <= 1)
      launch_gemv_k<EPI, 1, CHAIN>(a, c, st);
    else
      launch_gemv_k<EPI, 8, CHAIN>(a, c, st);
  } else if (a.x_f32) {
    launch_gemv_long<EPI, true>(a, st);
  } else {
    launch_gemv_long<EPI, false>(a, st);
  }
}

// Argument checks and GemvArgs shared by both GEMV entry points.
int32_t make_gemv_args(GemvArgs& a, const void* x, int32_t x_is_f32, int64_t x_stride, int32_t m, int32_t k,
                       const uint16_t* const* weights, int32_t n, int32_t epilogue, void* const* outputs,
                       int64_t out_stride, const uint16_t* addend, int64_t addend_stride, const uint16_t* rope_cos,
                       const uint16_t* rope_sin, int32_t head_dim, const char* who) {
  const std::string w(who);
  FL_REQUIRE(x && weights && outputs, w + ": null x/weights/outputs");
  FL_REQUIRE(m >= 1 && m <= kMaxM, w + ": rows of x must be 1..8");
  FL_REQUIRE(k > 0 && k % 8 == 0 && n > 0 && n % kRows == 0, w + ": K must be a multiple of 8, N of 4");
  FL_REQUIRE(x_stride >= k && out_stride >= n, w + ": bad row strides");
  FL_REQUIRE(reinterpret_cast<uintptr_t>(x) % 16 == 0 && (x_stride * (x_is_f32 ? 4 : 2)) % 16 == 0,
             w + ": x rows must be 16-byte aligned");
  FL_REQUIRE(epilogue >= kEpiPlain && epilogue <= kEpiRope, w + ": unknown epilogue");
  const int nmat = epilogue == kEpiRope ? 3 : (epilogue == kEpiSwiGlu ? 2 : 1);
  for (int i = 0; i < nmat; ++i) {
    FL_REQUIRE(weights[i] != nullptr && reinterpret_cast<uintptr_t>(weights[i]) % 16 == 0,
               w + ": weights must be non-null and 16-byte aligned");
    a.w[i] = weights[i];
  }
  const int nout = epilogue == kEpiRope ? 3 : 1;
  for (int i = 0; i < nout; ++i) {
    FL_REQUIRE(outputs[i] != nullptr, w + ": null output");
    a.y[i] = outputs[i];
  }
  if (epilogue == kEpiAdd) FL_REQUIRE(addend != nullptr && addend_stride >= n, w + ": bad addend");
  if (epilogue == kEpiSwiGlu) FL_REQUIRE(n % 2 == 0, w + ": SwiGLU needs an even N");
  if (epilogue == kEpiRope)
    FL_REQUIRE(rope_cos && rope_sin && head_dim >= 8 && head_dim % 8 == 0 && n % head_dim == 0,
               w + ": rope needs cos/sin tables and N a multiple of head_dim (multiple of 8)");
  a.x = x;
  a.x_f32 = x_is_f32 ? 1 : 0;
  a.x_stride = x_stride;
  a.M = m;
  a.K = k;
  a.N = n;
  a.y_stride = out_stride;
  a.addend = addend;
  a.addend_stride = addend_stride;
  a.cos = rope_cos;
  a.sin = rope_sin;
  a.head_dim = head_dim;
  return FL_OK;
}

}  // namespace
}  // namespace fl

extern "C" int32_t fl_gemv_bf16(const void* x, int32_t x_is_f32, int64_t x_stride, int32_t m, int32_t k,
                                const uint16_t* const* weights, int32_t n, int32_t epilogue, void* const* outputs,
                                int64_t out_stride, const uint16_t* addend, int64_t addend_stride,
                                const uint16_t* rope_cos, const uint16_t* rope_sin, int32_t head_dim, void* stream) {
  using namespace fl;
  clear_error();
  GemvArgs a{};
  const int32_t rc = make_gemv_args(a, x, x_is_f32, x_stride, m, k, weights, n, epilogue, outputs, out_stride, addend,
                                    addend_stride, rope_cos, rope_sin, head_dim, "fl_gemv_bf16");
  if (rc != FL_OK) return rc;
  hipStream_t st = static_cast<hipStream_t>(stream);
  const NormArgs none{};
  switch (epilogue) {
    case kEpiPlain: launch_gemv<kEpiPlain, false>(a, none, st); break;
    case kEpiF32: launch_gemv<kEpiF32, false>(a, none, st); break;
    case kEpiAdd: launch_gemv<kEpiAdd, false>(a, none, st); break;
    case kEpiSwiGlu: launch_gemv<kEpiSwiGlu, false>(a, none, st); break;
    default: launch_gemv<kEpiRope, false>(a, none, st); break;
  }
  FL_LAUNCH_CHECK("fl_gemv_bf16");
  return FL_OK;
}

extern "C" int32_t fl_gemv_bf16_chain(int32_t m, int32_t k, float eps, const uint16_t* x, const uint16_t* r,
                                      const uint16_t* w_a, const uint16_t* w_f, const uint16_t* w_b, uint16_t* h_out,
                                      int64_t stride, const uint16_t* const* weights, int32_t n, int32_t epilogue,
                                      void* const* outputs, int64_t out_stride, const uint16_t* addend,
                                      int64_t addend_stride, const uint16_t* rope_cos, const uint16_t* rope_sin,
                                      int32_t head_dim, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(r != nullptr, "fl_gemv_bf16_chain: null residual/input");
  FL_REQUIRE(k <= kChainMaxK && stride >= k && stride % 8 == 0,
             "fl_gemv_bf16_chain: K must be at most 4096 and the chain row stride a multiple of 8 >= K");
  FL_REQUIRE(x == nullptr || w_a != nullptr, "fl_gemv_bf16_chain: x needs its norm weight");
  for (const void* p : {static_cast<const void*>(x), static_cast<const void*>(r), static_cast<const void*>(w_a),
                        static_cast<const void*>(w_f), static_cast<const void*>(w_b), static_cast<const void*>(h_out)})
    FL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "fl_gemv_bf16_chain: every chain tensor must be 16-byte aligned");
  GemvArgs a{};
  // the GEMV's x is the chain output: its checks run on the residual row layout
  const int32_t rc = make_gemv_args(a, r, 0, stride, m, k, weights, n, epilogue, outputs, out_stride, addend,
                                    addend_stride, rope_cos, rope_sin, head_dim, "fl_gemv_bf16_chain");
  if (rc != FL_OK) return rc;
  const NormArgs c{k, eps, x, r, w_a, w_f, w_b, h_out, nullptr, stride};
  hipStream_t st = static_cast<hipStream_t>(stream);
  switch (epilogue) {
    case kEpiPlain: launch_gemv<kEpiPlain, true>(a, c, st); break;
    case kEpiF32: launch_gemv<kEpiF32, true>(a, c, st); break;
    case kEpiAdd: launch_gemv<kEpiAdd, true>(a, c, st); break;
    case kEpiSwiGlu: launch_gemv<kEpiSwiGlu, true>(a, c, st); break;
    default: launch_gemv<kEpiRope, true>(a, c, st); break;
  }
  FL_LAUNCH_CHECK("fl_gemv_bf16_chain");
  return FL_OK;
}

extern "C" int32_t fl_norm_chain(int32_t m, int32_t d, float eps, const uint16_t* x, const uint16_t* r,
                                 const uint16_t* w_a, const uint16_t* w_f, const uint16_t* w_b, uint16_t* h_out,
                                 uint16_t* z_out, int64_t stride, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(m >= 0 && d > 0 && d % 8 == 0 && d <= kNormThreads * kNormChunks * 8 && stride >= d && stride % 8 == 0,
             "fl_norm_chain: d must be a multiple of 8 up to 8192 and the row stride a multiple of 8");
  FL_REQUIRE(r != nullptr, "fl_norm_chain: null residual/input");
  FL_REQUIRE(x == nullptr || w_a != nullptr, "fl_norm_chain: x needs its norm weight");
  FL_REQUIRE(w_b == nullptr || z_out != nullptr, "fl_norm_chain: z needs an output");
  FL_REQUIRE(h_out != nullptr || z_out != nullptr, "fl_norm_chain: nothing to write");
  for (const void* p : {static_cast<const void*>(x), static_cast<const void*>(r), static_cast<const void*>(w_a),
                        static_cast<const void*>(w_f), static_cast<const void*>(w_b),
                        static_cast<const void*>(h_out), static_cast<const void*>(z_out)})
    FL_REQUIRE(reinterpret_cast<uintptr_t>(p) % 16 == 0, "fl_norm_chain: every tensor must be 16-byte aligned");
  if (m == 0) return FL_OK;
  NormArgs a{d, eps, x, r, w_a, w_f, w_b, h_out, z_out, stride};
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (d <= kNormThreads * 8)
    hipLaunchKernelGGL(norm_chain_kernel<1>, dim3(m), dim3(kNormThreads), 0, st, a);
  else if (d <= 2 * kNormThreads * 8)
    hipLaunchKernelGGL(norm_chain_kernel<2>, dim3(m), dim3(kNormThreads), 0, st, a);
  else
    hipLaunchKernelGGL(norm_chain_kernel<kNormChunks>, dim3(m), dim3(kNormThreads), 0, st, a);
  FL_LAUNCH_CHECK("fl_norm_chain");
  return FL_OK;
}

extern "C" int32_t fl_decode_inputs(const int64_t* tokens, const int64_t* positions, int32_t batch,
                                    const uint16_t* table, int64_t vocab, int32_t hidden, const void* inv_freq,
                                    int32_t freq_is_bf16, int32_t head_dim, uint16_t* h, uint16_t* rope_cos,
                                    uint16_t* rope_sin, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(tokens && positions && table && inv_freq && h && rope_cos && rope_sin, "fl_decode_inputs: null pointer");
  FL_REQUIRE(batch > 0 && vocab > 0 && hidden > 0 && hidden % 8 == 0 && head_dim > 0 && head_dim % 2 == 0,
             "fl_decode_inputs: bad sizes");
  FL_REQUIRE(reinterpret_cast<uintptr_t>(table) % 16 == 0 && reinterpret_cast<uintptr_t>(h) % 16 == 0,
             "fl_decode_inputs: the table and h must be 16-byte aligned");
  const InputArgs a{tokens, positions, table, vocab, hidden, head_dim / 2, inv_freq, freq_is_bf16, h, rope_cos, rope_sin};
  hipLaunchKernelGGL(decode_inputs_kernel, dim3(batch), dim3(kInputThreads), 0, static_cast<hipStream_t>(stream), a);
  FL_LAUNCH_CHECK("fl_decode_inputs");
  return FL_OK;
}

extern "C" int32_t fl_append_tails(const fl_cache_view* const* views, int32_t layers, const uint16_t* const* keys,
                                   const uint16_t* const* values, uint8_t* const* tail_active,
                                   int32_t* const* tail_tokens, void* stream) {
  using namespace fl;
  clear_error();
  FL_REQUIRE(views && keys && values && tail_active && tail_tokens && layers > 0, "fl_append_tail: null argument");
  for (int i = 0; i < layers; ++i) {
    FL_REQUIRE(views[i], "fl_append_tail: null argument");
    const fl_cache_view& v = *views[i];
    FL_REQUIRE(v.batch > 0 && v.heads > 0 && v.tail_capacity > 0 && v.tail_tokens, "fl_append_tail: bad view");
    FL_REQUIRE(v.batch == views[0]->batch && v.heads == views[0]->heads && v.tail_capacity == views[0]->tail_capacity,
               "fl_append_tails: the layers differ in batch, heads or tail capacity");
    FL_REQUIRE(tail_tokens[i] == v.tail_tokens, "fl_append_tail: tail_tokens must be the view's length array");
    for (int r = 4 * i; r < 4 * i + 4; ++r) {
      FL_REQUIRE(keys[r] && values[r] && v.tail_key[r & 3] && v.tail_value[r & 3], "fl_append_tail: null row or tail");
      FL_REQUIRE(reinterpret_cast<uintptr_t>(keys[r]) % 16 == 0 && reinterpret_cast<uintptr_t>(values[r]) % 16 == 0,
                 "fl_append_tail: rows must be 16-byte aligned");
    }
    FL_REQUIRE(tail_active[2 * i] && tail_active[2 * i + 1], "fl_append_tail: null tail_active");
  }
  for (int i0 = 0; i0 < layers; i0 += kAppendLayers) {
    const int n = layers - i0 < kAppendLayers ? layers - i0 : kAppendLayers;
    AppendArgs a{};
    a.heads = views[0]->heads;
    a.tail_capacity = views[0]->tail_capacity;
    for (int j = 0; j < n; ++j) {
      const int i = i0 + j;
      AppendLayer& l = a.layer[j];
      for (int r = 0; r < 4; ++r) {
        l.tail[r] = static_cast<uint16_t*>(views[i]->tail_key[r]);
        l.tail[4 + r] = static_cast<uint16_t*>(views[i]->tail_value[r]);
        l.rows[r] = keys[4 * i + r];
        l.rows[4 + r] = values[4 * i + r];
      }
      l.active[0] = tail_active[2 * i];
      l.active[1] = tail_active[2 * i + 1];
      l.tail_tokens = tail_tokens[i];
    }
    hipLaunchKernelGGL(append_tail_kernel, dim3(views[0]->batch, n), dim3(kAppendThreads), 0,
                       static_cast<hipStream_t>(stream), a);
    FL_LAUNCH_CHECK("fl_append_tail");
  }
  return FL_OK;
}

extern "C" int32_t fl_append_tail(const fl_cache_view* view, const uint16_t* const* keys,
                                  const uint16_t* const* values, uint8_t* const* tail_active,
                                  int32_t* tail_tokens, void* stream) {
  return fl_append_tails(&view, 1, keys, values, tail_active, &tail_tokens, stream);
}
