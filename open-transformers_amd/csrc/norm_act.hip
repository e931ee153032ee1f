// RMSNorm and SiLU for the decoder layer around the attention (BASELINE
// configuration 5).
//
// RMSNorm replaces repop.nn.rmsnorm.rms_norm (src/pretrain/model/modules/
// norm_repop.py:19-22; fp32 arithmetic, correctly rounded rsqrt, output in the
// input dtype, fp32 weight gradient: docs/MODEL_OP_DTYPE_TRACE.md:76-77,105).
// SiLU replaces repop.nn.activations.silu (ffn_repop.py; correctly rounded
// exp: MODEL_OP_DTYPE_TRACE.md:81,101).  Contract (binary32, RN):
//   fold32(f, n)  = partials p_c = serial fma over i = 32c .. 32c+31 from +0,
//                   then acc = +0, acc = acc + p_c for c ascending
//   RMSNorm fwd   ss = fold32(x_d * x_d), rstd = rsqrt(RN(RN(ss / D) + eps)),
//                 y_d = RN(RN(x_d * rstd) * w_d) (stored in the input dtype)
//   RMSNorm bwd   xh_d = RN(x_d * rstd), g_d = RN(dy_d * w_d),
//                 c = RN(fold32(g_d * xh_d) / D),
//                 dx_d = RN(rstd * RN(g_d - RN(xh_d * c)))
//                 dw_d = fold32 over rows r of dy_rd * xh_rd   (binary32)
//   SiLU fwd      d = RN(1 + exp(-x)), y = RN(x / d)
//   SiLU bwd      s = RN(1 / d), g = RN(s * RN(1 + RN(x * RN(1 - s)))),
//                 dx = RN(dy * g)
//   SwiGLU        gate, up = the two halves of each row of gu [rows, 2F]
//                 (ffn_repop.py:52-54: chunk(2, -1), silu(gate) * up):
//                 y = put(SiLU(gate)), h = put(RN(y * up));
//                 backward gy = put(RN(dh * up)), dgate = put(RN(gy * g)),
//                 dup = put(RN(dh * y)) into dgu [rows, 2F] (the halves of
//                 chunk's backward, which concatenates them)
// exp and rsqrt are correctly rounded; bf16 results are RNE of the binary32
// value.  One wave per row for the row reductions: lane c computes partial
// c (a serial fma chain), the partials are folded in order.
#include <initializer_list>
#include "otx_common.h"

namespace otx {

// 16 bytes of a T tensor: 8 bf16 or 4 binary32 elements.
template <typename T>
struct Act16 {
  static constexpr int N = 16 / sizeof(T);
  __device__ __forceinline__ static void load(const T* p, float (&v)[N]) {
    const uint4 w = *(const uint4*)p;
#pragma unroll
    for (int e = 0; e < N; e++) v[e] = Elem<T>::get(w, e);
  }
  __device__ __forceinline__ static void store(T* p, const float (&v)[N]) {
    uint4 w;
    uint32_t* wp = (uint32_t*)&w;
    if constexpr (sizeof(T) == 2) {
#pragma unroll
      for (int k = 0; k < 4; k++)
        wp[k] = (uint32_t)Elem<T>::put(v[2 * k]) | ((uint32_t)Elem<T>::put(v[2 * k + 1]) << 16);
    } else {
#pragma unroll
      for (int k = 0; k < 4; k++) wp[k] = __float_as_uint(v[k]);
    }
    *(uint4*)p = w;
  }
  __device__ __forceinline__ static float round(float v) {
    if constexpr (sizeof(T) == 2)
      return otx_bf16_to_f32(otx_f32_to_bf16(v));
    else
      return v;
  }
};

template <typename T>
struct Chunk32 {
  static constexpr int NV = 32 * (int)sizeof(T) / 16;  // 16-byte vectors per chunk
  __device__ __forceinline__ static void load(const T* p, float (&v)[32]) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      const uint4 w = reinterpret_cast<const uint4*>(p)[k];
#pragma unroll
      for (int e = 0; e < Elem<T>::VEC; e++) v[k * Elem<T>::VEC + e] = Elem<T>::get(w, e);
    }
  }
  __device__ __forceinline__ static void store(T* p, const float (&v)[32]) {
#pragma unroll
    for (int k = 0; k < NV; k++) {
      uint4 w;
      uint32_t* wp = reinterpret_cast<uint32_t*>(&w);
      if constexpr (sizeof(T) == 2) {
#pragma unroll
        for (int q = 0; q < 4; q++)
          wp[q] = (uint32_t)Elem<T>::put(v[8 * k + 2 * q]) | ((uint32_t)Elem<T>::put(v[8 * k + 2 * q + 1]) << 16);
      } else {
#pragma unroll
        for (int q = 0; q < 4; q++) wp[q] = __float_as_uint(v[4 * k + q]);
      }
      reinterpret_cast<uint4*>(p)[k] = w;
    }
  }
};

// Partials of fold32 over one row, v(c, e) the 32 terms' factors of chunk c: chunk c
// is computed by lane c % 64 into slot c / 64, +0 past the last chunk.
template <int SLOTS, typename F>
__device__ __forceinline__ void row_partials(int D, F&& chunk, float (&part)[SLOTS]) {
  const int L = threadIdx.x & 63;
#pragma unroll
  for (int s = 0; s < SLOTS; s++) {
    const int cidx = s * 64 + L;
    part[s] = cidx * 32 < D ? chunk(cidx) : 0.0f;
  }
}

// Ascending fold of the partials (chunk c in lane c % 64, slot c / 64); every
// lane ends with the same value.  Called by whole waves.  Lanes are read sixteen at a
// time, past the last chunk too: a partial there is +0, and the fold, begun at +0, is
// never -0, so adding it changes nothing.
template <int SLOTS>
__device__ __forceinline__ float fold_all(const float (&part)[SLOTS], int nch) {
  float acc = 0.0f;
#pragma unroll
  for (int s = 0; s < SLOTS; s++) {
    const int n = nch - 64 * s < 64 ? nch - 64 * s : 64;
    for (int l = 0; l < n; l += 16) {
#pragma unroll
      for (int u = 0; u < 16; u++)
        acc = acc + __int_as_float(__builtin_amdgcn_readlane(__float_as_int(part[s]), l + u));
    }
  }
  return acc;
}

// Elements p[0 .. 31], 16 bytes at a time where VEC says that p is aligned.
template <typename T, bool VEC>
__device__ __forceinline__ void load_chunk(const T* p, float (&v)[32]) {
  if constexpr (VEC) {
    Chunk32<T>::load(p, v);
  } else {
#pragma unroll
    for (int i = 0; i < 32; i++) v[i] = Elem<T>::ld(p + i);
  }
}

// One wave per row, any D = 32 n up to 64 * SLOTS chunks: the widths without a row-group
// form (VEC), and rows that are not 16-byte aligned.  Bound by the loads: a lane reads
// its chunk, and then the row again from the cache, 16 bytes at a time.  Measured at
// 8192 x 3008 bf16: forward 37.9 -> 22.0 us (4.5 TB/s), dx 45.5 -> 35.4 (a lane's chunk and
// the second pass were read 2 bytes at a time).
template <typename T, int SLOTS, bool VEC>
__global__ __launch_bounds__(256) void rmsnorm_fwd_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                          T* __restrict__ y, float* __restrict__ rstd_out, long rows,
                                                          int D, float eps) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int L = threadIdx.x & 63;
  const T* xr = x + row * D;
  float part[SLOTS];
  row_partials<SLOTS>(D, [&](int c) {
    float v[32], p = 0.0f;
    load_chunk<T, VEC>(xr + 32 * c, v);
#pragma unroll
    for (int i = 0; i < 32; i++) p = __builtin_fmaf(v[i], v[i], p);
    return p;
  }, part);
  const float ss = fold_all<SLOTS>(part, D / 32);
  const float mean = otx_div_rn(ss, (float)D);
  const float rstd = otx_rsqrtf(mean + eps);
  T* yr = y + row * D;
  if constexpr (VEC) {
    constexpr int N = Act16<T>::N;
    for (int d = L * N; d < D; d += 64 * N) {
      float v[N], wv[N];
      Act16<T>::load(xr + d, v);
      Act16<T>::load(w + d, wv);
#pragma unroll
      for (int e = 0; e < N; e++) v[e] = (v[e] * rstd) * wv[e];
      Act16<T>::store(yr + d, v);
    }
  } else {
    for (int d = L; d < D; d += 64) {
      const float xh = Elem<T>::ld(xr + d) * rstd;
      yr[d] = Elem<T>::put(xh * Elem<T>::ld(w + d));
    }
  }
  if (L == 0) rstd_out[row] = rstd;
}

template <typename T, int SLOTS, bool VEC>
__global__ __launch_bounds__(256) void rmsnorm_bwd_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                          const float* __restrict__ rstd_in,
                                                          const T* __restrict__ dy, T* __restrict__ dx, long rows,
                                                          int D) {
  const long row = (long)blockIdx.x * 4 + (threadIdx.x >> 6);
  if (row >= rows) return;
  const int L = threadIdx.x & 63;
  const T* xr = x + row * D;
  const T* dyr = dy + row * D;
  const float rstd = rstd_in[row];
  float part[SLOTS];
  row_partials<SLOTS>(D, [&](int c) {
    float xv[32], gv[32], wv[32], p = 0.0f;
    load_chunk<T, VEC>(xr + 32 * c, xv);
    load_chunk<T, VEC>(dyr + 32 * c, gv);
    load_chunk<T, VEC>(w + 32 * c, wv);
#pragma unroll
    for (int i = 0; i < 32; i++) p = __builtin_fmaf(gv[i] * wv[i], xv[i] * rstd, p);
    return p;
  }, part);
  const float cc = otx_div_rn(fold_all<SLOTS>(part, D / 32), (float)D);
  T* dxr = dx + row * D;
  if constexpr (VEC) {
    constexpr int N = Act16<T>::N;
    for (int d = L * N; d < D; d += 64 * N) {
      float xv[N], gv[N], wv[N];
      Act16<T>::load(xr + d, xv);
      Act16<T>::load(dyr + d, gv);
      Act16<T>::load(w + d, wv);
#pragma unroll
      for (int e = 0; e < N; e++) gv[e] = rstd * (gv[e] * wv[e] - (xv[e] * rstd) * cc);
      Act16<T>::store(dxr + d, gv);
    }
  } else {
    for (int d = L; d < D; d += 64) {
      const float xh = Elem<T>::ld(xr + d) * rstd;
      const float g = Elem<T>::ld(dyr + d) * Elem<T>::ld(w + d);
      dxr[d] = Elem<T>::put(rstd * (g - xh * cc));
    }
  }
}

// Row-group form for D = 32 G with G a power of two up to 64: lane L of a wave
// owns chunk c = L % G of row L / G (64 / G rows per wave) and reads its 32
// elements with 16-byte loads; the partials are folded in order with G
// shuffles inside the row's lane group.  Same arithmetic as the kernels above.
// Bound by HBM.  The forward's second pass walks the wave's 2048 elements side by side
// and reads x again from the cache: stores of a lane's own chunk left 64 bytes between
// lanes.  Measured, bf16: 8192 x 2048 19.4 -> 14.7 us (4.6 TB/s), 131072 x 128 18.4 ->
// 13.9.  The backward keeps its chunk (two tensors to read again: 21.8 us kept, 23.0
// re-read at 8192 x 2048).
// Ascending fold of the G partials of this lane's row group (every lane of the
// group ends with the same value).
template <int G>
__device__ __forceinline__ float fold_group(float p) {
  const int base = (threadIdx.x & 63) & ~(G - 1);
  float acc = 0.0f;
#pragma unroll
  for (int k = 0; k < G; k++) acc = acc + __shfl(p, base + k);
  return acc;
}

template <typename T, int G>
__global__ __launch_bounds__(256) void rmsnorm_fwd_rows_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                               T* __restrict__ y, float* __restrict__ rstd_out,
                                                               long rows, float eps) {
  constexpr int D = 32 * G, RPW = 64 / G, N = Act16<T>::N;
  const int L = threadIdx.x & 63, c = L % G;
  const long row0 = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW, row = row0 + L / G;
  const bool live = row < rows;
  float p = 0.0f;
  if (live) {
    float v[32];
    Chunk32<T>::load(x + row * D + 32 * c, v);
#pragma unroll
    for (int i = 0; i < 32; i++) p = __builtin_fmaf(v[i], v[i], p);
  }
  const float ss = fold_group<G>(p);
  const float rstd = otx_rsqrtf(otx_div_rn(ss, (float)D) + eps);
#pragma unroll
  for (int k = 0; k < 32 / N; k++) {
    const int i = (k * 64 + L) * N, r = i / D, d = i % D;  // element i of the wave's 2048
    const float rs = __shfl(rstd, r * G);
    if (row0 + r < rows) {
      float v[N], wv[N];
      Act16<T>::load(x + row0 * D + i, v);
      Act16<T>::load(w + d, wv);
#pragma unroll
      for (int e = 0; e < N; e++) v[e] = (v[e] * rs) * wv[e];
      Act16<T>::store(y + row0 * D + i, v);
    }
  }
  if (live && c == 0) rstd_out[row] = rstd;
}

template <typename T, int G>
__global__ __launch_bounds__(256) void rmsnorm_bwd_rows_kernel(const T* __restrict__ x, const T* __restrict__ w,
                                                               const float* __restrict__ rstd_in,
                                                               const T* __restrict__ dy, T* __restrict__ dx,
                                                               long rows) {
  constexpr int D = 32 * G, RPW = 64 / G;
  const int L = threadIdx.x & 63, c = L % G;
  const long row = ((long)blockIdx.x * 4 + (threadIdx.x >> 6)) * RPW + L / G;
  const bool live = row < rows;
  float xh[32], g[32];
  float rstd = 0.0f;
  if (live) {
    float wv[32];
    rstd = rstd_in[row];
    Chunk32<T>::load(x + row * D + 32 * c, xh);
    Chunk32<T>::load(dy + row * D + 32 * c, g);
    Chunk32<T>::load(w + 32 * c, wv);
#pragma unroll
    for (int i = 0; i < 32; i++) {
      xh[i] = xh[i] * rstd;
      g[i] = g[i] * wv[i];
    }
  } else {
#pragma unroll
    for (int i = 0; i < 32; i++) xh[i] = g[i] = 0.0f;
  }
  float p = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) p = __builtin_fmaf(g[i], xh[i], p);
  const float cc = otx_div_rn(fold_group<G>(p), (float)D);
  if (!live) return;
#pragma unroll
  for (int i = 0; i < 32; i++) g[i] = rstd * (g[i] - xh[i] * cc);
  Chunk32<T>::store(dx + row * D + 32 * c, g);
}

// dw partials: part[c][d] = serial fma over rows 32c .. 32c+31 of dy * xh.
template <typename T>
__global__ __launch_bounds__(256) void rmsnorm_dw_partial_kernel(const T* __restrict__ x,
                                                                 const float* __restrict__ rstd_in,
                                                                 const T* __restrict__ dy, float* __restrict__ part,
                                                                 long rows, int D) {
  const int d = blockIdx.x * 256 + threadIdx.x;
  const long cidx = blockIdx.y;
  if (d >= D) return;
  float acc = 0.0f;
  for (int i = 0; i < 32; i++) {
    const long r = cidx * 32 + i;
    const float xh = Elem<T>::ld(x + r * D + d) * rstd_in[r];
    acc = __builtin_fmaf(Elem<T>::ld(dy + r * D + d), xh, acc);
  }
  part[cidx * D + d] = acc;
}

// out[d] = serial fold over c ascending of part[c][d], from +0.  The chain of
// one column is inherently serial, so the work is arranged for its loads:
// a workgroup owns FC_W columns and stages FC_R partials of each through LDS
// with all 256 threads loading at once (one 16-byte load per partial row), so
// that a column of up to FC_R partials costs one memory round trip; then FC_W
// threads add them in order.
constexpr int FC_W = 4, FC_R = 4096;
__global__ __launch_bounds__(256) void fold_columns_kernel(const float* __restrict__ part, float* __restrict__ out,
                                                           long nch, int D) {
  __shared__ __align__(16) float tile[FC_R * FC_W];
  const int d0 = blockIdx.x * FC_W;
  const int t = threadIdx.x;
  float acc = 0.0f;
  for (long c0 = 0; c0 < nch; c0 += FC_R) {
    const int rows = nch - c0 < FC_R ? (int)(nch - c0) : FC_R;
    constexpr int PER = FC_R / 256;
    float4 v[PER];
#pragma unroll
    for (int k = 0; k < PER; k++) {
      const int r = t + 256 * k;
      v[k] = r < rows ? *reinterpret_cast<const float4*>(part + (c0 + r) * D + d0) : make_float4(0.f, 0.f, 0.f, 0.f);
    }
#pragma unroll
    for (int k = 0; k < PER; k++) reinterpret_cast<float4*>(tile)[t + 256 * k] = v[k];
    __syncthreads();
    if (t < FC_W) {
      int r = 0;
      for (; r + 16 <= rows; r += 16) {
        float q[16];
#pragma unroll
        for (int u = 0; u < 16; u++) q[u] = tile[(r + u) * FC_W + t];
#pragma unroll
        for (int u = 0; u < 16; u++) acc = acc + q[u];
      }
      for (; r < rows; r++) acc = acc + tile[r * FC_W + t];
    }
    __syncthreads();
  }
  if (t < FC_W) out[d0 + t] = acc;
}

// SiLU terms of N inputs: y = RN(x / d) and, for the backward, s = RN(1 / d),
// d = RN(1 + exp(-x)).  Both quotients go through one reciprocal of d, correctly
// rounded in the normal range; NaN (also the reciprocal of d = inf) and
// subnormal quotients take the division itself, behind a wave-uniform branch.  A
// zero y comes only from |x| so small that d = 2 exactly, where x * 0.5 rounds
// once, so zeros need no division.
template <int N, bool BACKWARD>
__device__ __forceinline__ void silu_terms(const float (&x)[N], float (&y)[N], float (&s)[N], const double* tab) {
  constexpr int UNSURE = 0x3 | 0x10 | 0x80;  // NaN, negative and positive subnormals (v_cmp_class)
  float d[N];
#pragma unroll
  for (int e = 0; e < N; e++) d[e] = -x[e];
  otx_exp_any_n<N>(d, tab);
  bool low = false;
#pragma unroll
  for (int e = 0; e < N; e++) {
    d[e] = 1.0f + d[e];
    const double r = otx_recip64_newton(d[e]);
    y[e] = (float)((double)x[e] * r);
    low = low || __builtin_amdgcn_classf(y[e], UNSURE);
    if constexpr (BACKWARD) {
      s[e] = (float)r;
      low = low || __builtin_amdgcn_classf(s[e], UNSURE);
    }
  }
  if (__builtin_expect(__ballot(low) != 0, 0)) {
#pragma unroll
    for (int e = 0; e < N; e++) {
      if (__builtin_amdgcn_classf(y[e], UNSURE)) y[e] = otx_div_rn(x[e], d[e]);
      if constexpr (BACKWARD)
        if (__builtin_amdgcn_classf(s[e], UNSURE)) s[e] = otx_div_rn(1.0f, d[e]);
    }
  }
}

// The activation kernels are bound by HBM once the exp and the quotients are
// short (about 30 vector instructions per element forward): a workgroup loads
// the exp table once and walks 16-byte vectors with the grid's stride.  Measured:
// SwiGLU forward and backward at 8192 x 5632 bf16 199 -> 146 us, 738 MB at
// 5.05 TB/s, the rate of a large copy (with otx_expf's degree-13 series, a division
// per quotient and one vector per thread it was bound by the vector ALU).
template <int N>
__device__ __forceinline__ void silu_one(const float (&x)[N], const float (&dy)[N], float (&r)[N], bool backward,
                                         const double* tab) {
  float y[N], s[N];
  if (!backward) {
    silu_terms<N, false>(x, r, s, tab);
    return;
  }
  silu_terms<N, true>(x, y, s, tab);
#pragma unroll
  for (int e = 0; e < N; e++) r[e] = dy[e] * (s[e] * (1.0f + x[e] * (1.0f - s[e])));
}

// vec: x, dy and out are 16-byte aligned; the n % N elements past the last whole
// vector, or all of them, go one by one.
template <typename T, bool BACKWARD>
__global__ __launch_bounds__(256) void silu_kernel(const T* __restrict__ x, const T* __restrict__ dy,
                                                   T* __restrict__ out, long n, int vec) {
  constexpr int N = Act16<T>::N;
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  otx_load_exp_table(tab);
  __syncthreads();
  const long i0 = (long)blockIdx.x * 256 + threadIdx.x, step = (long)gridDim.x * 256;
  const long nv = vec ? n / N : 0;
  for (long i = i0; i < nv; i += step) {
    float v[N], d[N], r[N];
    Act16<T>::load(x + i * N, v);
    if constexpr (BACKWARD) Act16<T>::load(dy + i * N, d);
    silu_one<N>(v, d, r, BACKWARD, tab);
    Act16<T>::store(out + i * N, r);
  }
  for (long i = nv * N + i0; i < n; i += step) {
    float v[1] = {Elem<T>::ld(x + i)}, d[1] = {0.0f}, r[1];
    if constexpr (BACKWARD) d[0] = Elem<T>::ld(dy + i);
    silu_one<1>(v, d, r, BACKWARD, tab);
    out[i] = Elem<T>::put(r[0]);
  }
}

// SwiGLU over rows of gu = [gate | up] (each F wide): one 16-byte vector of h
// (and of gate and up) at a time; cpr = F / N vectors per row.  I: the type of a
// vector's index (32 bits where they suffice: a division per vector).
template <typename T, typename I>
__global__ __launch_bounds__(256) void swiglu_fwd_kernel(const T* __restrict__ gu, T* __restrict__ h, I vectors,
                                                         I cpr) {
  constexpr int N = Act16<T>::N;
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  otx_load_exp_table(tab);
  __syncthreads();
  for (I g = (I)blockIdx.x * 256 + threadIdx.x; g < vectors; g += (I)gridDim.x * 256) {
    const I row = g / cpr;
    const T* gate = gu + ((long)row * cpr + g) * N;  // row 2 cpr + the vector's place g - row cpr
    float x[N], u[N], y[N], s[N];
    Act16<T>::load(gate, x);
    Act16<T>::load(gate + (long)cpr * N, u);
    silu_terms<N, false>(x, y, s, tab);
#pragma unroll
    for (int e = 0; e < N; e++) y[e] = Act16<T>::round(y[e]) * u[e];
    Act16<T>::store(h + (long)g * N, y);
  }
}

template <typename T, typename I>
__global__ __launch_bounds__(256) void swiglu_bwd_kernel(const T* __restrict__ gu, const T* __restrict__ dh,
                                                         T* __restrict__ dgu, I vectors, I cpr) {
  constexpr int N = Act16<T>::N;
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  otx_load_exp_table(tab);
  __syncthreads();
  for (I g = (I)blockIdx.x * 256 + threadIdx.x; g < vectors; g += (I)gridDim.x * 256) {
    const I row = g / cpr;
    const long at = ((long)row * cpr + g) * N;
    float x[N], u[N], d[N], y[N], s[N], dg[N], du[N];
    Act16<T>::load(gu + at, x);
    Act16<T>::load(gu + at + (long)cpr * N, u);
    Act16<T>::load(dh + (long)g * N, d);
    silu_terms<N, true>(x, y, s, tab);
#pragma unroll
    for (int e = 0; e < N; e++) {
      const float gy = Act16<T>::round(d[e] * u[e]);
      dg[e] = gy * (s[e] * (1.0f + x[e] * (1.0f - s[e])));
      du[e] = d[e] * Act16<T>::round(y[e]);
    }
    Act16<T>::store(dgu + at, dg);
    Act16<T>::store(dgu + at + (long)cpr * N, du);
  }
}

static bool aligned16p(const void* p) { return ((uintptr_t)p & 15u) == 0; }

// Rows of width D = 32 G (G a power of two up to 64) go to the row-group
// kernels when every row pointer is 16-byte aligned.
static int row_group(int D, std::initializer_list<const void*> ptrs) {
  if (D % 32) return 0;
  const int G = D / 32;
  if (G > 64 || (G & (G - 1))) return 0;
  for (const void* p : ptrs)
    if (!aligned16p(p)) return 0;
  return G;
}

template <typename T, int G>
static void launch_rows_fwd(const void* x, const void* w, void* y, float* rstd, long rows, float eps,
                            hipStream_t st) {
  const long per_block = 4L * (64 / G);
  hipLaunchKernelGGL((rmsnorm_fwd_rows_kernel<T, G>), dim3((unsigned)((rows + per_block - 1) / per_block)), dim3(256),
                     0, st, (const T*)x, (const T*)w, (T*)y, rstd, rows, eps);
}

template <typename T, int G>
static void launch_rows_bwd(const void* x, const void* w, const float* rstd, const void* dy, void* dx, long rows,
                            hipStream_t st) {
  const long per_block = 4L * (64 / G);
  hipLaunchKernelGGL((rmsnorm_bwd_rows_kernel<T, G>), dim3((unsigned)((rows + per_block - 1) / per_block)), dim3(256),
                     0, st, (const T*)x, (const T*)w, rstd, (const T*)dy, (T*)dx, rows);
}

template <typename T>
static bool launch_rows_fwd_any(int G, const void* x, const void* w, void* y, float* rstd, long rows, float eps,
                                hipStream_t st) {
  switch (G) {
    case 1: launch_rows_fwd<T, 1>(x, w, y, rstd, rows, eps, st); return true;
    case 2: launch_rows_fwd<T, 2>(x, w, y, rstd, rows, eps, st); return true;
    case 4: launch_rows_fwd<T, 4>(x, w, y, rstd, rows, eps, st); return true;
    case 8: launch_rows_fwd<T, 8>(x, w, y, rstd, rows, eps, st); return true;
    case 16: launch_rows_fwd<T, 16>(x, w, y, rstd, rows, eps, st); return true;
    case 32: launch_rows_fwd<T, 32>(x, w, y, rstd, rows, eps, st); return true;
    case 64: launch_rows_fwd<T, 64>(x, w, y, rstd, rows, eps, st); return true;
    default: return false;
  }
}

template <typename T>
static bool launch_rows_bwd_any(int G, const void* x, const void* w, const float* rstd, const void* dy, void* dx,
                                long rows, hipStream_t st) {
  switch (G) {
    case 1: launch_rows_bwd<T, 1>(x, w, rstd, dy, dx, rows, st); return true;
    case 2: launch_rows_bwd<T, 2>(x, w, rstd, dy, dx, rows, st); return true;
    case 4: launch_rows_bwd<T, 4>(x, w, rstd, dy, dx, rows, st); return true;
    case 8: launch_rows_bwd<T, 8>(x, w, rstd, dy, dx, rows, st); return true;
    case 16: launch_rows_bwd<T, 16>(x, w, rstd, dy, dx, rows, st); return true;
    case 32: launch_rows_bwd<T, 32>(x, w, rstd, dy, dx, rows, st); return true;
    case 64: launch_rows_bwd<T, 64>(x, w, rstd, dy, dx, rows, st); return true;
    default: return false;
  }
}

static bool all_aligned16(std::initializer_list<const void*> ptrs) {
  for (const void* p : ptrs)
    if (!aligned16p(p)) return false;
  return true;
}

// One slot of chunks per lane up to 2048 columns, four up to the largest width; 16-byte
// accesses where the base pointers are aligned (rows are: D is a multiple of 32).
template <typename T, bool VEC>
static void launch_wave_fwd(const void* x, const void* w, void* y, float* rstd, long rows, int D, float eps,
                            hipStream_t st) {
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  if (D <= 2048)
    hipLaunchKernelGGL((rmsnorm_fwd_kernel<T, 1, VEC>), grid, block, 0, st, (const T*)x, (const T*)w, (T*)y, rstd,
                       rows, D, eps);
  else
    hipLaunchKernelGGL((rmsnorm_fwd_kernel<T, 4, VEC>), grid, block, 0, st, (const T*)x, (const T*)w, (T*)y, rstd,
                       rows, D, eps);
}

template <typename T, bool VEC>
static void launch_wave_bwd(const void* x, const void* w, const float* rstd, const void* dy, void* dx, long rows,
                            int D, hipStream_t st) {
  const dim3 grid((unsigned)((rows + 3) / 4)), block(256);
  if (D <= 2048)
    hipLaunchKernelGGL((rmsnorm_bwd_kernel<T, 1, VEC>), grid, block, 0, st, (const T*)x, (const T*)w, rstd,
                       (const T*)dy, (T*)dx, rows, D);
  else
    hipLaunchKernelGGL((rmsnorm_bwd_kernel<T, 4, VEC>), grid, block, 0, st, (const T*)x, (const T*)w, rstd,
                       (const T*)dy, (T*)dx, rows, D);
}

template <typename T>
static hipError_t launch_rmsnorm_fwd_t(const void* x, const void* w, void* y, float* rstd, long rows, int D,
                                       float eps, hipStream_t st) {
  if (launch_rows_fwd_any<T>(row_group(D, {x, w, y}), x, w, y, rstd, rows, eps, st)) return hipGetLastError();
  if (all_aligned16({x, w, y}))
    launch_wave_fwd<T, true>(x, w, y, rstd, rows, D, eps, st);
  else
    launch_wave_fwd<T, false>(x, w, y, rstd, rows, D, eps, st);
  return hipGetLastError();
}

hipError_t launch_rmsnorm_fwd(int dtype, const void* x, const void* w, void* y, float* rstd, long rows, int D,
                              float eps, hipStream_t st) {
  return dtype == 1 ? launch_rmsnorm_fwd_t<uint16_t>(x, w, y, rstd, rows, D, eps, st)
                    : launch_rmsnorm_fwd_t<float>(x, w, y, rstd, rows, D, eps, st);
}

template <typename T>
static hipError_t launch_rmsnorm_bwd_t(const void* x, const void* w, const float* rstd, const void* dy, void* dx,
                                       float* dw, float* part, long rows, int D, hipStream_t st) {
  if (!launch_rows_bwd_any<T>(row_group(D, {x, w, dy, dx}), x, w, rstd, dy, dx, rows, st)) {
    if (all_aligned16({x, w, dy, dx}))
      launch_wave_bwd<T, true>(x, w, rstd, dy, dx, rows, D, st);
    else
      launch_wave_bwd<T, false>(x, w, rstd, dy, dx, rows, D, st);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  const long nch = rows / 32;
  hipLaunchKernelGGL((rmsnorm_dw_partial_kernel<T>), dim3((unsigned)((D + 255) / 256), (unsigned)nch), dim3(256), 0,
                     st, (const T*)x, rstd, (const T*)dy, part, rows, D);
  e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(fold_columns_kernel, dim3((unsigned)((D + FC_W - 1) / FC_W)), dim3(256), 0, st, part, dw, nch, D);
  return hipGetLastError();
}

hipError_t launch_rmsnorm_bwd(int dtype, const void* x, const void* w, const float* rstd, const void* dy, void* dx,
                              float* dw, float* part, long rows, int D, hipStream_t st) {
  return dtype == 1 ? launch_rmsnorm_bwd_t<uint16_t>(x, w, rstd, dy, dx, dw, part, rows, D, st)
                    : launch_rmsnorm_bwd_t<float>(x, w, rstd, dy, dx, dw, part, rows, D, st);
}

// Workgroups of a grid-stride kernel over n items of 256 threads: one item per
// thread up to eight workgroups per CU, then more items per thread (each
// workgroup pays the exp table once).
static unsigned act_grid(long n) {
  const long want = (n + 255) / 256, most = 8L * otx_cu_count();
  return (unsigned)(want < most ? (want > 0 ? want : 1) : most);
}

template <typename T, typename I>
static void launch_swiglu_t(int backward, const void* gu, const void* dh, void* out, long vectors, int cpr,
                            hipStream_t st) {
  const dim3 grid(act_grid(vectors)), block(256);
  if (backward)
    hipLaunchKernelGGL((swiglu_bwd_kernel<T, I>), grid, block, 0, st, (const T*)gu, (const T*)dh, (T*)out, (I)vectors,
                       (I)cpr);
  else
    hipLaunchKernelGGL((swiglu_fwd_kernel<T, I>), grid, block, 0, st, (const T*)gu, (T*)out, (I)vectors, (I)cpr);
}

hipError_t launch_swiglu(int dtype, int backward, const void* gu, const void* dh, void* out, long rows, int F,
                         hipStream_t st) {
  const int cpr = F / (dtype == 1 ? 8 : 4);
  const long vectors = rows * cpr;
  const bool small = vectors < (1L << 31);  // the grid's stride past the end still fits 32 unsigned bits
  if (dtype == 1)
    small ? launch_swiglu_t<uint16_t, uint32_t>(backward, gu, dh, out, vectors, cpr, st)
          : launch_swiglu_t<uint16_t, uint64_t>(backward, gu, dh, out, vectors, cpr, st);
  else
    small ? launch_swiglu_t<float, uint32_t>(backward, gu, dh, out, vectors, cpr, st)
          : launch_swiglu_t<float, uint64_t>(backward, gu, dh, out, vectors, cpr, st);
  return hipGetLastError();
}

template <typename T>
static void launch_silu_t(int backward, const void* x, const void* dy, void* out, long n, hipStream_t st) {
  const int vec = aligned16p(x) && aligned16p(out) && (!backward || aligned16p(dy));
  const dim3 grid(act_grid(vec ? (n + Act16<T>::N - 1) / Act16<T>::N : n)), block(256);
  if (backward)
    hipLaunchKernelGGL((silu_kernel<T, true>), grid, block, 0, st, (const T*)x, (const T*)dy, (T*)out, n, vec);
  else
    hipLaunchKernelGGL((silu_kernel<T, false>), grid, block, 0, st, (const T*)x, nullptr, (T*)out, n, vec);
}

hipError_t launch_silu(int dtype, int backward, const void* x, const void* dy, void* out, long n, hipStream_t st) {
  if (dtype == 1)
    launch_silu_t<uint16_t>(backward, x, dy, out, n, st);
  else
    launch_silu_t<float>(backward, x, dy, out, n, st);
  return hipGetLastError();
}

}  // namespace otx
