// Fused cross-entropy + z-loss for gfx950.
//
// Replaces pretrain.model.fused_loss.fused_ce_z_loss / _FusedCEZLoss
// (src/pretrain/model/fused_loss.py:40-120 of the reference) and the
// logsumexp of _z_loss_lse (src/pretrain/model/z_loss.py:53-66).  Contract
// (binary32, RN; exp and log correctly rounded):
//   fold(a[0..n))  recursive chunk-32 fold: partials of 32 consecutive values
//                  summed serially from +0, repeated on the partials until one
//                  value is left
//   per row        m = max x;  e_v = exp(RN(x_v - m));  Z = fold(e);
//                  lse = RN(log Z + m);  d = RN(lse - x_label);  q = RN(lse * lse)
//   forward        ce = RN(fold(d) / N);  z = coeff == 0 ? +0 : RN(f32(coeff) * RN(fold(q) / N))
//   backward       cs = RN(gce * f32(1/N));  c2 = f32(2 coeff / N);  coef = RN(RN(c2 * gz) * lse)
//                  sm = RN(e_v / Z);  g = RN(sm * cs);  coeff != 0: g = RN(g + RN(sm * coef));
//                  v == label: g = RN(g - cs);  stored in the logits dtype
// Layout: logits [N][V] row-major (bf16 or binary32), labels [N] int64,
// stats [5][N] binary32 = (m, Z, lse, d, q), loss [2] = (ce, z).
//
// Forward: one workgroup per row: the maximum, then exp and the partials of the
// 32-value chunks, then the fold of the partials in LDS.  Backward: elementwise
// from the stored (m, Z, lse).  Two forms of each.
//
// The general form (ce_fwd_kernel, ce_bwd_kernel) evaluates the correctly
// rounded exp of every logit, about 14 of its 20 vector instructions per logit.
//
// The table form (ce_fwd_table_kernel, ce_bwd_table_kernel) is for long rows of
// bf16.  Given the row's m (and Z, lse), exp(RN(x - m)) and the gradient are
// functions of the 16 bits of x alone, so a row of 128256 logits needs each
// function at no more than the 5632 values of the 22 binades [2^-14, 2^8) of
// either sign, the range of a language model's logits: they are evaluated into
// LDS once per row (the same operations, so the same bytes), and a logit then
// costs one LDS read and two or three vector instructions.  Groups of 2048 (or
// 512) logits that hold a value outside the window (zeros, tiny values, infinities,
// NaN) are evaluated directly.  Rows that are not 16-byte aligned and binary32 rows take
// the general form, and so do rows below CE_TABLE_MIN_V logits, which pay a table of the
// same size for less: forward and backward of 8192 rows, table against general form, V
// 4096 153 against 112 us, 8192 166 / 154, 12288 201 / 232, 16384 231 / 295, 32768 394 /
// 670, 128256 1421 / 2325.
// Measured at 8192 x 128256 bf16, forward and backward on one box, before the table form
// and now: logits N(0, 2^2) 1959 -> 1426 us (589 + 837; the backward's 4.2 GB at 5.0 TB/s);
// the last 256 of each row -inf 1965 -> 1427; half of each row -inf, in one run 2046 ->
// 1503, every second logit 1980 -> 1880; zeros 3976 -> 1778; N(0, 1e-3^2), a value outside
// the window in most groups, 1911 -> 1963 (943 + 968 -> 834 + 1129).  The general forward
// against one lane per chunk in memory: 4096 x 50257 bf16 637 -> 300 us, 2000 x 5003 bf16
// 99 -> 34 us, 4096 x 128256 binary32 940 -> 761 us.
#include "otx_common.h"

namespace otx {

constexpr int CE_LT = 512;               // threads per row in the table form's forward
constexpr int CE_MT = 1024;              // threads of the final means
constexpr int CE_MAX_CHUNKS = 4096;      // 32-logit chunks per row: V <= 131072
constexpr int CE_TPB = 32;               // backward: 2048-logit tiles per workgroup and row
constexpr int CE_TABLE_MIN_V = 16384;
constexpr int CE_WIN_LO = 113 << 7;      // bf16 magnitude bits of 2^-14
constexpr int CE_WIN_N = 22 * 128;       // bf16 magnitudes in the window
constexpr int CE_TAB_N = 2 * CE_WIN_N;   // entry 2 (magnitude - CE_WIN_LO) + sign

typedef unsigned short u16x2 __attribute__((ext_vector_type(2)));
typedef short i16x2 __attribute__((ext_vector_type(2)));

// Recursive chunk-32 fold of n values in LDS.  Values live at ce_slot(i), one pad
// word per 32, so that 32 threads reading a chunk each hit distinct banks; the slots
// of the last chunk past n hold +0, which leaves a partial sum unchanged (a sum from
// +0 is never -0).  Every thread of the block calls it with the same n <= 32 * 32 * 32
// (three levels); the partials of the levels go to b; all threads see the result.
__device__ __forceinline__ int ce_slot(int i) { return i + (i >> 5); }
__device__ __forceinline__ float ce_fold_chunk(const float* a, int c) {
  float v[32];
#pragma unroll
  for (int i = 0; i < 32; i++) v[i] = a[33 * c + i];
  float s = 0.0f;
#pragma unroll
  for (int i = 0; i < 32; i++) s = s + v[i];
  return s;
}
// Zeros the slots of the last chunk past n (before the values' barrier).
__device__ __forceinline__ void ce_pad(float* a, int n) {
  const int i = n + (int)threadIdx.x;
  if (i < (n + 31) / 32 * 32) a[ce_slot(i)] = 0.0f;
}
__device__ float ce_block_fold(const float* a, float* b, int n) {
  while (true) {  // one level per round; a level's partials are padded like the values
    const int parts = (n + 31) / 32;
    for (int c = threadIdx.x; c < (parts + 31) / 32 * 32; c += blockDim.x)
      b[ce_slot(c)] = c < parts ? ce_fold_chunk(a, c) : 0.0f;
    __syncthreads();
    if (parts == 1) return b[0];
    a = b;
    b += ce_slot((parts + 31) / 32 * 32);
    n = parts;
  }
}
// Words of LDS for the partials of n values (all levels).
constexpr int ce_fold_words(int n) {
  int w = 0;
  while (n > 1) {
    n = (n + 31) / 32;
    w += (n + 31) / 32 * 33;
  }
  return w + 33;
}

// The row's statistics from its fold Z and maximum m, by one thread.
template <typename T>
__device__ __forceinline__ void ce_store_stats(const T* row, long n, long N, int V, long lab, float m, float Z,
                                               float* __restrict__ stats) {
  const float lse = otx_logf(Z) + m;
  const float d = lab >= 0 && lab < V ? lse - Elem<T>::ld(row + lab) : __builtin_nanf("");
  stats[n] = m;
  stats[N + n] = Z;
  stats[2 * N + n] = lse;
  stats[3 * N + n] = d;
  stats[4 * N + n] = lse * lse;
}

// v[j] = exp(v[j]) for v[j] = RN(x - m), with NaN (x or m not finite) put back where it
// was: the softmax path for m the row's maximum (v[j] <= 0), or, with ANY, the one for
// either sign (the backward's m is the caller's, and a logit may lie above it).
template <int N, int NB = 8, bool ANY = false>
__device__ __forceinline__ void ce_exp_n(float (&v)[N], const double* tab) {
  float mx = v[0];
#pragma unroll
  for (int j = 1; j + 1 < N; j += 2) mx = otx_max2p(otx_max2p(mx, v[j]), v[j + 1]);
  mx = otx_max2p(mx, v[N - 1]);
  uint32_t nan = 0;
  if (__builtin_expect(__ballot(mx != mx) != 0, 0)) {
#pragma unroll
    for (int j = 0; j < N; j++) nan |= v[j] != v[j] ? 1u << j : 0u;
  }
  if constexpr (ANY)
    otx_exp_any_n<N, NB>(v, tab);
  else
    otx_exp_n<N, false, NB>(v, tab);
  if (__builtin_expect(__ballot(nan != 0) != 0, 0)) {
#pragma unroll
    for (int j = 0; j < N; j++) v[j] = nan >> j & 1 ? __builtin_nanf("") : v[j];
  }
}

// ---- general forward ----
// A wave takes tiles of 2048 consecutive logits (64 chunks).  A tile is loaded with
// its lanes side by side in memory (16 bytes per lane, or element by element for rows
// that are not 16-byte aligned); the exps go through the wave's own 8 KiB of LDS, 16-byte
// units swizzled by chunk, and lane c adds chunk c serially.  W waves per row.
template <typename T, bool VEC>
struct CeTile {
  static constexpr int N = 16 / sizeof(T);  // logits per vector
  static constexpr int PL = VEC ? N : 1;    // logits per load
  static constexpr int NL = 16 / PL;        // loads per lane and half tile
  // The lane's logits of half h of tile t as binary32, -inf past the end of the row.
  __device__ __forceinline__ static void load(const T* row, int t, int h, int V, int L, float (&x)[16]) {
    const T* p = row + 2048 * t + 1024 * h;  // wave-uniform
    const int left = V - (2048 * t + 1024 * h);
    if (left >= 1024) {
#pragma unroll
      for (int k = 0; k < NL; k++) get(p, (64 * k + L) * PL, x, k);
    } else {
#pragma unroll
      for (int k = 0; k < NL; k++) {
        const int i = (64 * k + L) * PL;  // VEC: V is a multiple of N, so a vector lies inside the row or past it
#pragma unroll
        for (int e = 0; e < PL; e++) x[k * PL + e] = -__builtin_inff();
        if (i < left) get(p, i, x, k);
      }
    }
  }
  __device__ __forceinline__ static void get(const T* p, int i, float (&x)[16], int k) {
    if constexpr (VEC) {
      const uint4 w = *reinterpret_cast<const uint4*>(p + i);
#pragma unroll
      for (int e = 0; e < N; e++) x[k * N + e] = Elem<T>::get(w, e);
    } else {
      x[k] = Elem<T>::ld(p + i);
    }
  }
  // Word of logit j of chunk c in the tile's LDS.
  __device__ __forceinline__ static int word(int c, int j) { return 32 * c + 4 * ((j >> 2) ^ (c & 7)) + (j & 3); }
  __device__ __forceinline__ static void put(float* lds, int h, int L, const float (&e)[16]) {
#pragma unroll
    for (int k = 0; k < NL; k++) {
      const int i = 1024 * h + (64 * k + L) * PL;
      if constexpr (VEC) {
#pragma unroll
        for (int u = 0; u < N; u += 4)
          *reinterpret_cast<float4*>(lds + word(i >> 5, (i & 31) + u)) =
              make_float4(e[k * N + u], e[k * N + u + 1], e[k * N + u + 2], e[k * N + u + 3]);
      } else {
        lds[word(i >> 5, i & 31)] = e[k];
      }
    }
  }
};

template <typename T, bool VEC, int W>
__global__ __launch_bounds__(64 * W) void ce_fwd_kernel(const T* __restrict__ logits,
                                                        const int64_t* __restrict__ labels, long N, int V,
                                                        float* __restrict__ stats) {
  constexpr int CHUNKS = W == 1 ? 64 : W == 4 ? 512 : CE_MAX_CHUNKS;
  using Tile = CeTile<T, VEC>;
  __shared__ __align__(16) double tab[OTX_EXP_LE0_TAB_N];
  __shared__ __align__(16) float tile[W][2048];
  __shared__ float pa[CHUNKS / 32 * 33];
  __shared__ float pb[ce_fold_words(CHUNKS)];
  __shared__ float wmax[W];
  const int t = threadIdx.x, wave = t >> 6, L = t & 63;
  otx_load_exp_table(tab);
  const int nch = (V + 31) / 32, tiles = (V + 2047) / 2048;
  for (long n = blockIdx.x; n < N; n += gridDim.x) {
    const T* row = logits + (size_t)n * V;
    float mx = -__builtin_inff();
    for (int k = 2 * wave; k < 2 * tiles; k += k & 1 ? 2 * W - 1 : 1) {  // both halves of every tile of the wave
      float x[16];
      Tile::load(row, k >> 1, k & 1, V, L, x);
#pragma unroll
      for (int i = 0; i < 16; i++) mx = x[i] > mx ? x[i] : mx;
    }
    // block maximum (exact in any order)
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float y = __shfl_xor(mx, o);
      mx = y > mx ? y : mx;
    }
    if (L == 0) wmax[wave] = mx;
    ce_pad(pa, nch);
    __syncthreads();
    float m = wmax[0];
#pragma unroll
    for (int w = 1; w < W; w++) m = wmax[w] > m ? wmax[w] : m;
    for (int k = wave; k < tiles; k += W) {
#pragma unroll 1
      for (int h = 0; h < 2; h++) {
        float x[16];
        Tile::load(row, k, h, V, L, x);
#pragma unroll
        for (int i = 0; i < 16; i++) x[i] = x[i] - m;
        ce_exp_n<16, 4>(x, tab);
        Tile::put(tile[wave], h, L, x);
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      float s = 0.0f;
#pragma unroll
      for (int u = 0; u < 8; u++) {
        const float4 v = *reinterpret_cast<const float4*>(&tile[wave][Tile::word(L, 4 * u)]);
        s = s + v.x; s = s + v.y; s = s + v.z; s = s + v.w;  // logits past the end add +0
      }
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      __builtin_amdgcn_wave_barrier();
      if (64 * k + L < nch) pa[ce_slot(64 * k + L)] = s;
    }
    __syncthreads();
    const float Z = ce_block_fold(pa, pb, nch);
    if (t == 0) ce_store_stats<T>(row, n, N, V, labels[n], m, Z, stats);
    __syncthreads();  // the next row rewrites the partials
  }
}

// ---- table form of the forward ----
// (magnitude, sign) of the two bf16 of a word, each as magnitude * 2 + sign: ordered by
// magnitude, and the table's order.
__device__ __forceinline__ uint32_t ce_rot(uint32_t w) {
  const u16x2 v = __builtin_bit_cast(u16x2, w);
  return __builtin_bit_cast(uint32_t, (u16x2)((v << 1) | (v >> 15)));
}
__device__ __forceinline__ uint32_t ce_unrot(uint32_t r) {
  const u16x2 v = __builtin_bit_cast(u16x2, r);
  return __builtin_bit_cast(uint32_t, (u16x2)((v >> 1) | (v << 15)));
}
// Byte address of entry (half of the word r) * SIZE from the entry of rotated bits 0,
// which lies at byte -2 * CE_WIN_LO * SIZE: one instruction.
template <int HALF, int SIZE>
__device__ __forceinline__ uint32_t ce_entry(uint32_t r, uint32_t base) {
  uint32_t a;
  if constexpr (HALF)
    asm("v_mad_u32_u16 %0, %1, %3, %2 op_sel:[1,0,0,0]" : "=v"(a) : "v"(r), "s"(base), "n"(SIZE));
  else
    asm("v_mad_u32_u16 %0, %1, %3, %2" : "=v"(a) : "v"(r), "s"(base), "n"(SIZE));
  return a;
}
__device__ __forceinline__ u16x2 ce_min2(u16x2 a, u16x2 b) { return __builtin_elementwise_min(a, b); }
__device__ __forceinline__ u16x2 ce_max2(u16x2 a, u16x2 b) { return __builtin_elementwise_max(a, b); }
__device__ __forceinline__ uint32_t ce_lo_min(u16x2 v) { return v.x < v.y ? v.x : v.y; }
__device__ __forceinline__ uint32_t ce_hi_max(u16x2 v) { return v.x > v.y ? v.x : v.y; }
__device__ __forceinline__ float ce_bf16(uint32_t bits) { return __uint_as_float(bits << 16); }
// The bf16 value of table entry i.
__device__ __forceinline__ float ce_tab_x(int i) {
  return ce_bf16((uint32_t)(CE_WIN_LO + (i >> 1)) | ((uint32_t)(i & 1) << 15));
}

// One row per workgroup, read twice: for the maximum, then for the chunk partials,
// when most of it still lies in the last-level cache (three workgroups per CU hold
// 200 MB of rows).  Several workgroups per CU, because a row's phases (stream, table,
// LDS reads, fold) leave the memory or the LDS idle in turn: a form that kept the
// row in registers, one 1024-thread workgroup per CU with the next row's loads issued
// as the chunks were consumed, took 713 us against 600.
__global__ __launch_bounds__(CE_LT) void ce_fwd_table_kernel(const uint16_t* __restrict__ logits, long N, int V,
                                                             float* __restrict__ stats) {
  __shared__ __align__(16) float etab[CE_TAB_N];
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  __shared__ float pa[CE_MAX_CHUNKS / 32 * 33];
  __shared__ float pb[ce_fold_words(CE_MAX_CHUNKS)];
  __shared__ int wred[CE_LT / 64];
  __shared__ float wmax[CE_LT / 64];
  const int t = threadIdx.x, wave = t >> 6, L = t & 63;
  otx_load_exp_table(tab);
  const int nch = (V + 31) / 32, nv = V / 8;
  const uint32_t base = otx_lds_addr(etab) - 8u * CE_WIN_LO;
  const long n = blockIdx.x;
  const uint16_t* row = logits + (size_t)n * V;
  const uint4* vrow = reinterpret_cast<const uint4*>(row);
  // ---- maximum: the largest of the bits as signed integers, if that is a positive number; a
  // row without one, or with a positive NaN (passed over as in the general form), is
  // compared as binary32 ----
  i16x2 smax = {-32768, -32768};
#pragma unroll 8
  for (int i = t; i < nv; i += CE_LT) {
    const uint4 u = vrow[i];
    const uint32_t w[4] = {u.x, u.y, u.z, u.w};
#pragma unroll
    for (int x = 0; x < 4; x++) smax = __builtin_elementwise_max(smax, __builtin_bit_cast(i16x2, w[x]));
  }
  int sm = smax.x > smax.y ? smax.x : smax.y;
#pragma unroll
  for (int o = 32; o >= 1; o >>= 1) {
    const int a = __shfl_xor(sm, o);
    sm = a > sm ? a : sm;
  }
  if (L == 0) wred[wave] = sm;
  ce_pad(pa, nch);
  __syncthreads();
#pragma unroll
  for (int w = 0; w < CE_LT / 64; w++) sm = wred[w] > sm ? wred[w] : sm;
  float m = ce_bf16((uint32_t)sm);
  if (__builtin_expect(sm < 0 || sm > 0x7f80, 0)) {
    float mx = -__builtin_inff();
    for (int i = t; i < V; i += CE_LT) {
      const float x = Elem<uint16_t>::ld(row + i);
      mx = x > mx ? x : mx;
    }
#pragma unroll
    for (int o = 32; o >= 1; o >>= 1) {
      const float y = __shfl_xor(mx, o);
      mx = y > mx ? y : mx;
    }
    if (L == 0) wmax[wave] = mx;
    __syncthreads();
    m = wmax[0];
#pragma unroll
    for (int w = 1; w < CE_LT / 64; w++) m = wmax[w] > m ? wmax[w] : m;
  }
  // ---- exp(RN(x - m)) of every value of the window (values above m do not occur) ----
#pragma unroll 1
  for (int i = t; i < CE_TAB_N; i += 4 * CE_LT) {
    float e[4];
#pragma unroll
    for (int j = 0; j < 4; j++) {
      const float x = ce_tab_x(i + j * CE_LT);
      e[j] = x <= m ? x - m : -__builtin_inff();
    }
    otx_exp_n<4>(e, tab);
#pragma unroll
    for (int j = 0; j < 4; j++)
      if (i + j * CE_LT < CE_TAB_N) etab[i + j * CE_LT] = e[j];
  }
  __syncthreads();
  // ---- the chunk partials, summed serially from +0 ----
  uint4 nxt[4];
  const auto load = [&](int c) {
#pragma unroll
    for (int x = 0; x < 4; x++) {  // past the end: -inf
      nxt[x] = make_uint4(0xff80ff80u, 0xff80ff80u, 0xff80ff80u, 0xff80ff80u);
      if (4 * c + x < nv) nxt[x] = vrow[4 * c + x];
    }
  };
  load(t);
  for (int c = t; c < nch; c += CE_LT) {
    uint32_t r[16];
    u16x2 cmin = {0xffff, 0xffff}, cmax = {0, 0};
#pragma unroll
    for (int x = 0; x < 4; x++) {
      r[4 * x] = nxt[x].x; r[4 * x + 1] = nxt[x].y; r[4 * x + 2] = nxt[x].z; r[4 * x + 3] = nxt[x].w;
    }
    load(c + CE_LT);
#pragma unroll
    for (int x = 0; x < 16; x++) {
      r[x] = ce_rot(r[x]);
      cmin = ce_min2(cmin, __builtin_bit_cast(u16x2, r[x]));
      cmax = ce_max2(cmax, __builtin_bit_cast(u16x2, r[x]));
    }
    const bool in = ce_lo_min(cmin) >= 2 * CE_WIN_LO && ce_hi_max(cmax) < 2 * (CE_WIN_LO + CE_WIN_N);
    float s = 0.0f;
    if (__builtin_expect(__ballot(!in) == 0, 1)) {
#pragma unroll
      for (int x = 0; x < 16; x++) {
        s = s + *reinterpret_cast<const __attribute__((address_space(3))) float*>(ce_entry<0, 4>(r[x], base));
        s = s + *reinterpret_cast<const __attribute__((address_space(3))) float*>(ce_entry<1, 4>(r[x], base));
      }
    } else {
#pragma unroll
      for (int h = 0; h < 4; h++) {
        float e[8];
#pragma unroll
        for (int x = 0; x < 4; x++) {
          const uint32_t w = ce_unrot(r[4 * h + x]);
          e[2 * x] = __uint_as_float(w << 16) - m;
          e[2 * x + 1] = __uint_as_float(w & 0xffff0000u) - m;
        }
        ce_exp_n<8, 4>(e, tab);
#pragma unroll
        for (int i = 0; i < 8; i++) s = s + e[i];
      }
    }
    pa[ce_slot(c)] = s;
  }
  __syncthreads();
  const float Z = ce_block_fold(pa, pb, nch);
  if (t == 0) {
    stats[n] = m;
    stats[N + n] = Z;
  }
}

// lse, d and q of the rows whose m and Z the table form wrote (there, the log's
// constants would take the registers that hold a row).
__global__ __launch_bounds__(256) void ce_stats_kernel(const uint16_t* __restrict__ logits,
                                                       const int64_t* __restrict__ labels, long N, int V,
                                                       float* __restrict__ stats) {
  const long n = (long)blockIdx.x * 256 + threadIdx.x;
  if (n < N) ce_store_stats<uint16_t>(logits + (size_t)n * V, n, N, V, labels[n], stats[n], stats[N + n], stats);
}

// ce and z from the per-row d and q (one workgroup, a half of it for each; N <= 32 * 8192).
__global__ __launch_bounds__(CE_MT) void ce_mean_kernel(const float* __restrict__ stats, long N, float coeff32,
                                                        int has_coeff, float* __restrict__ loss) {
  __shared__ float pa[2][8192 / 32 * 33];
  __shared__ float pb[ce_fold_words(8192)];
  const int parts = (int)((N + 31) / 32);
  const int which = threadIdx.x / (CE_MT / 2);
  const float* a = stats + (3 + which) * N;
  for (int c = threadIdx.x % (CE_MT / 2); c < (parts + 31) / 32 * 32; c += CE_MT / 2) {
    float v[32];
#pragma unroll
    for (int i = 0; i < 32; i++) v[i] = 32L * c + i < N ? a[32L * c + i] : 0.0f;
    float s = 0.0f;
#pragma unroll
    for (int i = 0; i < 32; i++) s = s + v[i];
    pa[which][ce_slot(c)] = s;
  }
  __syncthreads();
  float f[2];
#pragma unroll 1
  for (int w = 0; w < 2; w++) {
    f[w] = ce_block_fold(pa[w], pb, parts);
    __syncthreads();
  }
  if (threadIdx.x == 0) {
    loss[0] = otx_div_rn(f[0], (float)N);
    loss[1] = has_coeff ? coeff32 * otx_div_rn(f[1], (float)N) : 0.0f;
  }
}

// ---- backward: gradient of ce * gce + z * gz with respect to the logits (gloss = {gce, gz}) ----
struct CeRow {
  float m, Z, cs, coef;
  double rz;
  long lab;
};
__device__ __forceinline__ CeRow ce_row(const float* __restrict__ stats, const float* __restrict__ gloss,
                                        const int64_t* __restrict__ labels, long N, long n, float inv_n, float c2) {
  CeRow r;
  r.m = stats[n];
  r.Z = stats[N + n];
  r.cs = gloss[0] * inv_n;
  r.coef = (c2 * gloss[1]) * stats[2 * N + n];
  r.lab = labels[n];
  r.rz = otx_recip64(r.Z);
  return r;
}
// g[i] = the gradient, but for the label's - cs, from e[i] = exp(RN(x_i - m)).  sm = RN(e / Z)
// goes through one binary64 reciprocal of Z (rz), with the bytes of
// otx_div_by_recip_checked: correctly rounded in the normal range; below it, where
// a quotient can be a midpoint exactly, and for NaN, the division itself, behind a
// wave-uniform branch.  (An e of zero needs none: 0 * rz is what 0 / Z is.)
template <int N>
__device__ __forceinline__ void ce_grad(const float (&e)[N], const CeRow& r, int has_coeff, float (&g)[N]) {
  bool low = false;
#pragma unroll
  for (int i = 0; i < N; i++) {
    g[i] = otx_div_by_recip(e[i], r.rz);
    low = low || (!(g[i] >= 0x1p-126f) && e[i] != 0.0f);
  }
  if (__builtin_expect(__ballot(low) != 0, 0)) {
#pragma unroll
    for (int i = 0; i < N; i++)
      if (!(g[i] >= 0x1p-126f) && e[i] != 0.0f) g[i] = otx_div_rn(e[i], r.Z);
  }
#pragma unroll
  for (int i = 0; i < N; i++) {
    const float sm = g[i];
    g[i] = sm * r.cs;
    if (has_coeff) g[i] = g[i] + sm * r.coef;
  }
}

// General form: 8 logits per thread, in 16-byte vectors of a tile, or one by one in rows
// that are not 16-byte aligned (the lanes side by side in memory either way).  A workgroup takes CE_TPB tiles of 2048 logits of
// a row at a time (one exp table for all of its rows).
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void ce_bwd_kernel(const T* __restrict__ logits, const int64_t* __restrict__ labels,
                                                     const float* __restrict__ stats, const float* __restrict__ gloss,
                                                     long N, int V, int tiles, float inv_n, float c2, int has_coeff,
                                                     T* __restrict__ grad) {
  constexpr int PL = VEC ? 16 / sizeof(T) : 1;  // logits per load
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  otx_load_exp_table(tab);
  __syncthreads();
  const int groups = (tiles + CE_TPB - 1) / CE_TPB;
  for (long it = blockIdx.x; it < N * groups; it += gridDim.x) {
    const long n = it / groups;
    const int t0 = (int)(it % groups) * CE_TPB;
    const CeRow row = ce_row(stats, gloss, labels, N, n, inv_n, c2);
    const T* src = logits + (size_t)n * V;
    T* dst = grad + (size_t)n * V;
    for (int k = t0; k < t0 + CE_TPB && k < tiles; k++) {
      if (2048 * k + (int)(threadIdx.x & ~63u) * PL >= V) break;  // this wave is past the row
      const auto at = [&](int i) { return 2048 * k + (256 * (i / PL) + (int)threadIdx.x) * PL + i % PL; };
      float e[8];
#pragma unroll
      for (int q = 0; q < 8; q += PL) {
        if constexpr (VEC) {  // V is a multiple of PL: a vector lies inside the row or past it
          const uint32_t ninf = sizeof(T) == 2 ? 0xff80ff80u : 0xff800000u;
          uint4 u = make_uint4(ninf, ninf, ninf, ninf);
          if (at(q) < V) u = *reinterpret_cast<const uint4*>(src + at(q));
#pragma unroll
          for (int i = 0; i < PL; i++) e[q + i] = Elem<T>::get(u, i);
        } else {
          e[q] = at(q) < V ? Elem<T>::ld(src + at(q)) : -__builtin_inff();
        }
      }
#pragma unroll
      for (int i = 0; i < 8; i++) e[i] = e[i] - row.m;
      ce_exp_n<8, 8, true>(e, tab);
      float g[8];
      ce_grad<8>(e, row, has_coeff, g);
#pragma unroll
      for (int i = 0; i < 8; i++)
        if (at(i) == row.lab) g[i] = g[i] - row.cs;
#pragma unroll
      for (int q = 0; q < 8; q += PL) {
        if (at(q) >= V) continue;
        if constexpr (VEC) {
          uint4 u;
          uint32_t* w = reinterpret_cast<uint32_t*>(&u);
#pragma unroll
          for (int i = 0; i < 4; i++) {
            if constexpr (sizeof(T) == 2)
              w[i] = (uint32_t)otx_f32_to_bf16(g[2 * i]) | ((uint32_t)otx_f32_to_bf16(g[2 * i + 1]) << 16);
            else
              w[i] = __float_as_uint(g[q + i]);
          }
          *reinterpret_cast<uint4*>(dst + at(q)) = u;
        } else {
          dst[at(q)] = Elem<T>::put(g[q]);
        }
      }
    }
  }
}

// Table form: one row per workgroup, the window's gradients as bf16 in LDS.  A wave
// whose 512 logits hold the label or a value outside the window evaluates them directly.
__global__ __launch_bounds__(256) void ce_bwd_table_kernel(const uint16_t* __restrict__ logits,
                                                           const int64_t* __restrict__ labels,
                                                           const float* __restrict__ stats,
                                                           const float* __restrict__ gloss, long N, int V, float inv_n,
                                                           float c2, int has_coeff, uint16_t* __restrict__ grad) {
  __shared__ __align__(16) uint16_t gtab[CE_TAB_N];
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  otx_load_exp_table(tab);
  __syncthreads();
  const long n = blockIdx.x;
  const int t = threadIdx.x;
  const CeRow row = ce_row(stats, gloss, labels, N, n, inv_n, c2);
  for (int i0 = t; i0 < CE_TAB_N; i0 += 8 * 256) {
    float e[8], g[8];
#pragma unroll
    for (int j = 0; j < 8; j++) e[j] = ce_tab_x(i0 + 256 * j) - row.m;
    ce_exp_n<8, 8, true>(e, tab);
    ce_grad<8>(e, row, has_coeff, g);
#pragma unroll
    for (int j = 0; j < 8; j++)
      if (i0 + 256 * j < CE_TAB_N) gtab[i0 + 256 * j] = otx_f32_to_bf16(g[j]);
  }
  __syncthreads();
  const uint32_t base = otx_lds_addr(gtab) - 4u * CE_WIN_LO;
  const uint4* src = reinterpret_cast<const uint4*>(logits + (size_t)n * V);
  uint4* dst = reinterpret_cast<uint4*>(grad + (size_t)n * V);
  const int nv = V / 8;
#pragma unroll 4
  for (int i = t; i < nv; i += 256) {
    const uint4 u = src[i];
    uint32_t w[4] = {u.x, u.y, u.z, u.w}, r[4];
    u16x2 lo = {0xffff, 0xffff}, hi = {0, 0};
#pragma unroll
    for (int x = 0; x < 4; x++) {
      r[x] = ce_rot(w[x]);
      lo = ce_min2(lo, __builtin_bit_cast(u16x2, r[x]));
      hi = ce_max2(hi, __builtin_bit_cast(u16x2, r[x]));
    }
    const bool direct = !(ce_lo_min(lo) >= 2 * CE_WIN_LO && ce_hi_max(hi) < 2 * (CE_WIN_LO + CE_WIN_N)) ||
                        (row.lab >= 8L * i && row.lab < 8L * i + 8);
    if (__builtin_expect(__ballot(direct) == 0, 1)) {
#pragma unroll
      for (int x = 0; x < 4; x++) {
        const uint32_t a =
            *reinterpret_cast<const __attribute__((address_space(3))) uint16_t*>(ce_entry<0, 2>(r[x], base));
        const uint32_t b =
            *reinterpret_cast<const __attribute__((address_space(3))) uint16_t*>(ce_entry<1, 2>(r[x], base));
        w[x] = a | (b << 16);
      }
    } else {
      float e[8], g[8];
#pragma unroll
      for (int j = 0; j < 8; j++) e[j] = Elem<uint16_t>::get(u, j) - row.m;
      ce_exp_n<8, 4, true>(e, tab);
      ce_grad<8>(e, row, has_coeff, g);
#pragma unroll
      for (int j = 0; j < 8; j++)
        if (8L * i + j == row.lab) g[j] = g[j] - row.cs;
#pragma unroll
      for (int x = 0; x < 4; x++)
        w[x] = (uint32_t)otx_f32_to_bf16(g[2 * x]) | ((uint32_t)otx_f32_to_bf16(g[2 * x + 1]) << 16);
    }
    dst[i] = make_uint4(w[0], w[1], w[2], w[3]);
  }
}

// Largest vocabulary of the forward's LDS partials.
int ce_max_vocab(int) { return 32 * CE_MAX_CHUNKS; }

static bool ce_table(int dtype, int V, int vec) { return dtype == 1 && vec && V >= CE_TABLE_MIN_V; }

template <typename T, bool VEC>
static void launch_ce_fwd_t(const void* logits, const int64_t* labels, long N, int V, float* stats, hipStream_t st) {
  // waves per row: one per 2048-logit tile of the row, rounded to the forms 1, 4 and 16;
  // a workgroup goes on to further rows past eight rounds of the device
  const long most = 8L * otx_cu_count();
#define OTX_CE_FWD(W)                                                                                            \
  hipLaunchKernelGGL((ce_fwd_kernel<T, VEC, W>), dim3((unsigned)(N < most * (16 / W) ? N : most * (16 / W))),     \
                     dim3(64 * W), 0, st, (const T*)logits, labels, N, V, stats)
  if (V <= 2048) OTX_CE_FWD(1);
  else if (V <= 16384) OTX_CE_FWD(4);
  else OTX_CE_FWD(16);
#undef OTX_CE_FWD
}

hipError_t launch_ce_fwd(int dtype, const void* logits, const int64_t* labels, long N, int V, int vec, float coeff32,
                         int has_coeff, float* stats, float* loss, hipStream_t st) {
  if (ce_table(dtype, V, vec)) {
    hipLaunchKernelGGL(ce_fwd_table_kernel, dim3((unsigned)N), dim3(CE_LT), 0, st, (const uint16_t*)logits, N, V,
                       stats);
    const hipError_t e = hipGetLastError();
    if (e != hipSuccess) return e;
    hipLaunchKernelGGL(ce_stats_kernel, dim3((unsigned)((N + 255) / 256)), dim3(256), 0, st, (const uint16_t*)logits,
                       labels, N, V, stats);
  } else if (dtype == 1) {
    vec ? launch_ce_fwd_t<uint16_t, true>(logits, labels, N, V, stats, st)
        : launch_ce_fwd_t<uint16_t, false>(logits, labels, N, V, stats, st);
  } else {
    vec ? launch_ce_fwd_t<float, true>(logits, labels, N, V, stats, st)
        : launch_ce_fwd_t<float, false>(logits, labels, N, V, stats, st);
  }
  hipError_t e = hipGetLastError();
  if (e != hipSuccess) return e;
  hipLaunchKernelGGL(ce_mean_kernel, dim3(1), dim3(CE_MT), 0, st, (const float*)stats, N, coeff32, has_coeff, loss);
  return hipGetLastError();
}

hipError_t launch_ce_bwd(int dtype, const void* logits, const int64_t* labels, const float* stats,
                         const float* gloss, long N, int V, int vec, float inv_n, float c2, int has_coeff, void* grad,
                         hipStream_t st) {
  if (ce_table(dtype, V, vec)) {
    hipLaunchKernelGGL(ce_bwd_table_kernel, dim3((unsigned)N), dim3(256), 0, st, (const uint16_t*)logits, labels,
                       stats, gloss, N, V, inv_n, c2, has_coeff, (uint16_t*)grad);
    return hipGetLastError();
  }
  const int tiles = (V + 2047) / 2048;
  const long items = N * ((tiles + CE_TPB - 1) / CE_TPB), most = 16L * otx_cu_count();
  const dim3 grid((unsigned)(items < most ? items : most)), block(256);
#define OTX_CE_BWD(T, VEC)                                                                                     \
  hipLaunchKernelGGL((ce_bwd_kernel<T, VEC>), grid, block, 0, st, (const T*)logits, labels, stats, gloss, N, V, \
                     tiles, inv_n, c2, has_coeff, (T*)grad)
  if (dtype == 1) {
    if (vec) OTX_CE_BWD(uint16_t, true); else OTX_CE_BWD(uint16_t, false);
  } else {
    if (vec) OTX_CE_BWD(float, true); else OTX_CE_BWD(float, false);
  }
#undef OTX_CE_BWD
  return hipGetLastError();
}

}  // namespace otx
