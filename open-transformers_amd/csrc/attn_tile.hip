// Causal / sliding-window attention on 16 x 16 tiles that four waves share.
//
// The kernels of attn_fwd.hip and attn_bwd.hip give one wave a whole 32-row
// block: a matrix instruction of 64 cycles advances a block's fold by one term,
// and a wave's 64-key step is one serial chain of products, softmax and
// products.  That fills the device once there are several blocks per SIMD, but
// a small grid waits for that chain, and binary32 operands (twice the registers
// and LDS of bf16) left one wave per SIMD with nothing to hide it behind.
//
// Here a workgroup's four waves share one block.  v_mfma_f32_16x16x4_f32 is four
// serial fmas per output in 32 cycles (checked against the serial fold), so a
// 16 x 16 tile advances one term in 8 cycles, and each wave takes a quarter of
// the keys for the scores and a quarter of the width for the outputs.  A wave
// holds few registers (the operands that stay, 16 rows of them, and its
// accumulators), so several workgroups share a CU and one's softmax runs under
// another's products.  The bytes are those of the other kernels: the same folds
// in the same order.
//
// Lane L = 16 g + c.  One instruction: A lane supplies row c, term g; B lane
// column c, term g; result register r holds row 4 g + r, column c.  Operands
// whose terms run along a row in memory are loaded as four consecutive terms per
// lane and transposed between the four lane groups (otx_transpose4); operands
// whose terms run across rows are loaded as they are.  A result whose rows
// become the next product's terms goes through LDS in the order [term / 16]
// [term % 4][column][term / 4 % 4], where both the four-byte writes and the
// 16-byte reads are free of bank conflicts.
#include "otx_common.h"

namespace otx {

typedef float f32x4 __attribute__((ext_vector_type(4)));
typedef int i32x4 __attribute__((ext_vector_type(4)));

__device__ __forceinline__ f32x4 otx_mfma_k4(float a, float b, f32x4 c) {
  return __builtin_amdgcn_mfma_f32_16x16x4f32(a, b, c, 0, 0, 0);
}

// a[j] of lane group g  ->  a[t] holds what group t had in a[g] (4 x 4 transpose between the lane groups).
__device__ __forceinline__ void otx_swap_rows16(float& x, float& y) {
  auto r = __builtin_amdgcn_permlane16_swap(__float_as_uint(x), __float_as_uint(y), false, false);
  x = __uint_as_float(r[0]);
  y = __uint_as_float(r[1]);
}
__device__ __forceinline__ void otx_transpose4(float (&a)[4]) {
  otx_swap_rows16(a[0], a[1]);
  otx_swap_rows16(a[2], a[3]);
  otx_swap_halves(a[0], a[2]);
  otx_swap_halves(a[1], a[3]);
}

// Four (or N = 1, 2) consecutive elements as loaded, and their binary32 values.
template <typename T, int N> struct TileRaw;
template <> struct TileRaw<float, 4> { typedef float4 V; };
template <> struct TileRaw<float, 2> { typedef float2 V; };
template <> struct TileRaw<float, 1> { typedef float V; };
template <> struct TileRaw<uint16_t, 4> { typedef uint2 V; };
template <> struct TileRaw<uint16_t, 2> { typedef uint32_t V; };
template <> struct TileRaw<uint16_t, 1> { typedef uint16_t V; };
template <typename T, int N>
__device__ __forceinline__ typename TileRaw<T, N>::V tile_load(const T* p) {
  return *reinterpret_cast<const typename TileRaw<T, N>::V*>(p);
}
__device__ __forceinline__ float bf_lo(uint32_t w) { return __uint_as_float(w << 16); }
__device__ __forceinline__ float bf_hi(uint32_t w) { return __uint_as_float(w & 0xffff0000u); }
__device__ __forceinline__ void tile_get(float4 v, float (&a)[4]) { a[0] = v.x; a[1] = v.y; a[2] = v.z; a[3] = v.w; }
__device__ __forceinline__ void tile_get(uint2 v, float (&a)[4]) {
  a[0] = bf_lo(v.x); a[1] = bf_hi(v.x); a[2] = bf_lo(v.y); a[3] = bf_hi(v.y);
}
__device__ __forceinline__ void tile_get(float2 v, float (&a)[2]) { a[0] = v.x; a[1] = v.y; }
__device__ __forceinline__ void tile_get(uint32_t v, float (&a)[2]) { a[0] = bf_lo(v); a[1] = bf_hi(v); }
__device__ __forceinline__ void tile_get(float v, float (&a)[1]) { a[0] = v; }
__device__ __forceinline__ void tile_get(uint16_t v, float (&a)[1]) { a[0] = bf_lo(v); }

// N (4 or 8) consecutive binary32 values to storage, N * sizeof(T) bytes aligned.
template <int N>
__device__ __forceinline__ void tile_store(float* p, const float (&x)[N]) {
#pragma unroll
  for (int i = 0; i < N; i += 4) *reinterpret_cast<float4*>(p + i) = make_float4(x[i], x[i + 1], x[i + 2], x[i + 3]);
}
__device__ __forceinline__ uint32_t bf_pair(float a, float b) {
  return (uint32_t)otx_f32_to_bf16(a) | (uint32_t)otx_f32_to_bf16(b) << 16;
}
__device__ __forceinline__ void tile_store(uint16_t* p, const float (&x)[4]) {
  *reinterpret_cast<uint2*>(p) = make_uint2(bf_pair(x[0], x[1]), bf_pair(x[2], x[3]));
}
__device__ __forceinline__ void tile_store(uint16_t* p, const float (&x)[8]) {
  *reinterpret_cast<uint4*>(p) =
      make_uint4(bf_pair(x[0], x[1]), bf_pair(x[2], x[3]), bf_pair(x[4], x[5]), bf_pair(x[6], x[7]));
}

// Maximum over the four lane groups, in every lane (NaN-propagating like otx_max32).
__device__ __forceinline__ float tile_max_groups(float v) {
  float x = v, y = v;
  otx_swap_rows16(x, y);
  x = otx_max2p(x, y);
  y = x;
  otx_swap_halves(x, y);
  return otx_max2p(x, y);
}

__device__ __attribute__((noinline)) float otx_logf_tile_call(float x) { return otx_logf(x); }

// Forward.  A workgroup owns 16 NQ consecutive queries of one head and walks its
// key blocks in ascending pairs, two barriers per pair:
//   S^T: wave w takes keys 16 w .. 16 w + 15 of the 64 (A = K rows straight from
//        global memory, loaded one pair ahead; B = the workgroup's Q, in registers);
//   block maxima across the waves through LDS, then each lane's 4 NQ exps;
//   O^T: wave w takes d = w D/4 .. (A = V straight from global memory, loaded
//        before the scores; B = the probabilities of all four waves, from LDS);
//   the running sum l (a serial fold over the 64 keys) is kept in LDS and
//   advanced by one wave per pair, the four waves in turn.
// The fp32 matrix instructions and the vector unit take turns, so what is left
// beside 32 cycles per product is vector work: K's transposes (one per product
// pair), 4 NQ exps per lane, the sums.  4 heads x 256 x 64 in binary32: 36 -> 14
// us; 16 heads x 1024 x 128 in bf16: 166 -> 76 us (its products alone: 14 us).
// I8 (int8-PV): the probabilities also go to LDS as bytes with their block's step
// and O^T += dequant(V^T P^T) takes one v_mfma_i32_16x16x32_i8 per 16 columns and
// key block (integer sums, so the order of its keys does not matter): 134 -> 69 us.
template <typename T, int D, int NQ, bool I8 = false>
__global__ __launch_bounds__(256, 2) void attn_fwd_tile_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, T* __restrict__ o,
    float* __restrict__ lse, int B, int H, int Hkv, int S, int window, float sigma, int order,
    float* __restrict__ scache, const int8_t* __restrict__ qvt, const float* __restrict__ vstep) {
  constexpr int KS = D / 4;   // four-term steps of a score
  constexpr int NT = D / 64;  // 16-wide output tiles per wave
  constexpr int UPB = 2 / NQ; // workgroups per query block
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  __shared__ float4 Pb[NQ][4][64];
  __shared__ float Mx[4][16 * NQ];
  __shared__ float Ls[16 * NQ];
  __shared__ uint2 Pq[I8 ? 2 : 1][NQ][16][4];  // int8 probabilities [key block][.][query][8 keys]
  __shared__ float Sp[2][16 * NQ];             // and their steps

  const int nqt = S / OTX_BLK, units = nqt * UPB, BH = B * H;
  const int bid = blockIdx.x + gridDim.x * blockIdx.y;
  if (bid >= units * BH) return;  // a grid of several rows (see fwd_tile_grid) may end in spare workgroups
  int unit, bh;
  if (order == 0) {  // longest key ranges first, heads fastest
    unit = units - 1 - bid / BH;
    bh = bid % BH;
  } else {
    unit = bid % units;
    bh = bid / units;
  }
  const int b = bh / H, h = bh % H, gk = h / (H / Hkv);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), L = threadIdx.x & 63, g = L >> 4, c = L & 15;
  const int qt = unit / UPB, q0 = unit * 16 * NQ;
  const T* kg = k + ((size_t)b * Hkv + gk) * S * D;
  const T* vg = v + ((size_t)b * Hkv + gk) * S * D;

  otx_load_exp_table(tab);
  if (threadIdx.x < 16 * NQ) Ls[threadIdx.x] = 0.0f;

  typedef typename TileRaw<T, 4>::V R4;
  typedef typename TileRaw<T, NT>::V RN;
  float qr[NQ][KS];
#pragma unroll
  for (int n = 0; n < NQ; n++) {
    const T* src = q + ((size_t)bh * S + q0 + 16 * n + c) * D + 4 * g;
#pragma unroll
    for (int u = 0; u < KS / 4; u++) {
      float a[4];
      tile_get(tile_load<T, 4>(src + 16 * u), a);
      otx_transpose4(a);
#pragma unroll
      for (int e = 0; e < 4; e++) qr[n][4 * u + e] = a[e];
    }
  }
  const int lo = otx_kblock_lo(qt, window);
  const int edge = window > 0 ? qt - window / OTX_BLK : -1;  // key block at the window's lower edge
  const T* ksrc = kg + (size_t)(16 * w + c) * D + 4 * g;
  const T* vsrc = vg + (size_t)g * D + w * (D / 4) + NT * c;
  R4 kraw[KS / 4];
  // a block past the diagonal is not used: the last one is loaded again, so that every pass defines kraw
  auto load_k = [&](int ka) {
    const int kb = ka + (w >> 1) < qt ? ka + (w >> 1) : qt;
    const T* p = ksrc + (size_t)(kb - (w >> 1)) * OTX_BLK * D;
#pragma unroll
    for (int u = 0; u < KS / 4; u++) kraw[u] = tile_load<T, 4>(p + 16 * u);
  };
  load_k(lo);

  float m[NQ];
  f32x4 acc[NQ][NT];
#pragma unroll
  for (int n = 0; n < NQ; n++) {
    m[n] = -__builtin_inff();
#pragma unroll
    for (int j = 0; j < NT; j++) acc[n][j] = f32x4{};
  }
  __syncthreads();

  int turn = 0;
  for (int ka = lo; ka <= qt; ka += 2, turn = (turn + 1) & 3) {
    const bool doB = ka + 1 <= qt;
    const bool wact = w < 2 || doB;
    RN vraw[I8 ? 1 : 16];
    uint2 vq[2][NT];
    float4 vst[2][NT];
    if constexpr (I8) {  // d = w D/4 + 16 j + row; a block past the diagonal is not used
#pragma unroll
      for (int x = 0; x < 2; x++) {
        const size_t blk = ((size_t)b * Hkv + gk) * nqt + (ka + x < qt ? ka + x : qt);
        const uint2* qp = reinterpret_cast<const uint2*>(qvt + (blk * D + w * (D / 4) + c) * 32 + 8 * g);
        const float4* sp = reinterpret_cast<const float4*>(vstep + blk * D + w * (D / 4) + 4 * g);
#pragma unroll
        for (int j = 0; j < NT; j++) {
          vq[x][j] = qp[64 * j];
          vst[x][j] = sp[4 * j];
        }
      }
    } else {
      const T* p = vsrc + (size_t)ka * OTX_BLK * D;
#pragma unroll
      for (int t = 0; t < 8; t++) vraw[t] = tile_load<T, NT>(p + (size_t)4 * t * D);
      if (doB) {
#pragma unroll
        for (int t = 8; t < 16; t++) vraw[t] = tile_load<T, NT>(p + (size_t)4 * t * D);
      }
    }
    float s[(I8 ? 5 : 4) * NQ];  // with I8 the last NQ become the largest probability of this wave's block
    if (wact) {
      f32x4 sa[NQ];
#pragma unroll
      for (int n = 0; n < NQ; n++) sa[n] = f32x4{};
#pragma unroll
      for (int u = 0; u < KS / 4; u++) {
        float a[4];
        tile_get(kraw[u], a);
        otx_transpose4(a);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int n = 0; n < NQ; n++) sa[n] = otx_mfma_k4(a[e], qr[n][4 * u + e], sa[n]);
      }
      load_k(ka + 2);
      const int kblk = ka + (w >> 1), j0 = kblk * OTX_BLK + 16 * (w & 1) + 4 * g;
      const bool need_mask = kblk == qt || kblk == edge;
#pragma unroll
      for (int n = 0; n < NQ; n++)
#pragma unroll
        for (int r = 0; r < 4; r++) {
          s[4 * n + r] = sa[n][r] * sigma;
          if (need_mask)
            s[4 * n + r] = otx_masked(q0 + 16 * n + c, j0 + r, window) ? -__builtin_inff() : s[4 * n + r];
        }
      if constexpr (sizeof(T) == 2) {
        if (scache != nullptr) {  // the tile [key j][query] of attn_fwd_bf16_kernel's score cache
          float* tile = scache + (((long)bh * otx_tile_offset(nqt, window) + otx_tile_offset(qt, window) +
                                   (kblk - lo)) << 10);
#pragma unroll
          for (int n = 0; n < NQ; n++)
#pragma unroll
            for (int r = 0; r < 4; r++)
              tile[(16 * (w & 1) + 4 * g + r) * 32 + (q0 & 31) + 16 * n + c] = s[4 * n + r];
        }
      }
    } else {
#pragma unroll
      for (int x = 0; x < 4 * NQ; x++) s[x] = -__builtin_inff();
    }
    float mx[NQ];
#pragma unroll
    for (int n = 0; n < NQ; n++)
      mx[n] = tile_max_groups(otx_max2p(otx_max2p(otx_max2p(s[4 * n], s[4 * n + 1]), s[4 * n + 2]), s[4 * n + 3]));
    if (L < 16 * NQ) Mx[w][L] = NQ == 2 && g == 1 ? mx[NQ - 1] : mx[0];
    __syncthreads();
    float al_a[NQ], al_b[NQ];
    {
      float al[2 * NQ], ma[NQ], mbn[NQ];
      bool moved = false;
#pragma unroll
      for (int n = 0; n < NQ; n++) {
        const float mba = otx_max2p(Mx[0][16 * n + c], Mx[1][16 * n + c]);
        const float mbb = otx_max2p(Mx[2][16 * n + c], Mx[3][16 * n + c]);
        ma[n] = otx_max_update(mba, m[n]);
        mbn[n] = doB ? otx_max_update(mbb, ma[n]) : ma[n];
        if constexpr (I8) s[4 * NQ + n] = w < 2 ? mba : mbb;
        al[2 * n] = ma[n] == m[n] ? 0.0f : m[n] - ma[n];
        al[2 * n + 1] = mbn[n] == ma[n] ? 0.0f : ma[n] - mbn[n];
        moved = moved || ma[n] != m[n] || mbn[n] != ma[n];
      }
      if (__any(moved)) otx_exp_n<2 * NQ>(al, tab);  // otherwise every factor is 1
#pragma unroll
      for (int n = 0; n < NQ; n++) {
        al_a[n] = ma[n] == m[n] ? 1.0f : al[2 * n];
        al_b[n] = mbn[n] == ma[n] ? 1.0f : al[2 * n + 1];
        const float mref = w < 2 ? ma[n] : mbn[n];
        const float moff = mref != -__builtin_inff() ? mref : __builtin_inff();
#pragma unroll
        for (int r = 0; r < 4; r++) s[4 * n + r] = s[4 * n + r] - moff;
        if constexpr (I8) s[4 * NQ + n] = s[4 * NQ + n] - moff;
        m[n] = mbn[n];
      }
    }
    otx_exp_n<(I8 ? 5 : 4) * NQ, false, I8 ? 5 : 4>(s, tab);
    if constexpr (I8) {
      // The block's largest probability is the exp of its largest score: the difference and the correctly
      // rounded exp are both monotone (a NaN score makes every probability of the row +0, as in the other form).
      // Step and bytes as in attn_fwd_bf16_kernel, four keys per lane.
#pragma unroll
      for (int n = 0; n < NQ; n++) {
        const float pmax = s[4 * NQ + n];
        float inv = 0.0f, sp = 0.0f;
        if (pmax > 0.0f) {
          inv = otx_div_rn(127.0f, pmax);
          sp = otx_div_by_recip(pmax, OTX_RECIP64_127);
        }
        uint32_t word = 0;
#pragma unroll
        for (int e = 0; e < 4; e++) word = __builtin_amdgcn_cvt_pk_u8_f32(s[4 * n + e] * inv, e, word);
        reinterpret_cast<uint32_t*>(&Pq[w >> 1][n][c][0])[4 * (w & 1) + g] = word & 0x7f7f7f7fu;
        if (!(w & 1) && g == n) Sp[w >> 1][16 * n + c] = sp;
      }
    }
#pragma unroll
    for (int n = 0; n < NQ; n++)
#pragma unroll
      for (int r = 0; r < 4; r++) reinterpret_cast<float*>(&Pb[n][w][16 * r + c])[g] = s[4 * n + r];
    __syncthreads();
    if (w == turn) {  // l = RN(l * alpha), then + p ascending, per block
      const int n = NQ == 2 ? g & 1 : 0;
      float l = Ls[16 * n + c] * (NQ == 2 && n ? al_a[NQ - 1] : al_a[0]);
#pragma unroll
      for (int t4 = 0; t4 < 4; t4++) {
        if (t4 >= 2 && !doB) break;
        if (t4 == 2) l = l * (NQ == 2 && n ? al_b[NQ - 1] : al_b[0]);
        float x[4][4];
#pragma unroll
        for (int i = 0; i < 4; i++) tile_get(Pb[n][t4][16 * i + c], x[i]);
#pragma unroll
        for (int e = 0; e < 4; e++)
#pragma unroll
          for (int i = 0; i < 4; i++) l = l + x[i][e];
      }
      if (L < 16 * NQ) Ls[L] = l;
    }
    auto scale = [&](const float (&al)[NQ]) {
      bool any = false;
#pragma unroll
      for (int n = 0; n < NQ; n++) any = any || al[n] != 1.0f;
      if (__any(any)) {
#pragma unroll
        for (int n = 0; n < NQ; n++)
#pragma unroll
          for (int j = 0; j < NT; j++)
#pragma unroll
            for (int r = 0; r < 4; r++) acc[n][j][r] = acc[n][j][r] * al[n];
      }
    };
    auto fold = [&](int t4) {  // 16 keys
      float p[NQ][4];
#pragma unroll
      for (int n = 0; n < NQ; n++) tile_get(Pb[n][t4][L], p[n]);
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float x[NT];
        tile_get(vraw[4 * t4 + e], x);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int n = 0; n < NQ; n++) acc[n][j] = otx_mfma_k4(x[j], p[n][e], acc[n][j]);
      }
    };
    if constexpr (I8) {
      auto fold8 = [&](int x) {
#pragma unroll
        for (int n = 0; n < NQ; n++) {
          const uint2 pb = Pq[x][n][c][g];
          const float sp = Sp[x][16 * n + c];
#pragma unroll
          for (int j = 0; j < NT; j++) {
            const i32x4 pv = __builtin_amdgcn_mfma_i32_16x16x32_i8(__builtin_bit_cast(long, vq[x][j]),
                                                                   __builtin_bit_cast(long, pb), i32x4{}, 0, 0, 0);
            float st[4];
            tile_get(vst[x][j], st);
#pragma unroll
            for (int r = 0; r < 4; r++) acc[n][j][r] = __builtin_fmaf((float)pv[r] * st[r], sp, acc[n][j][r]);
          }
        }
      };
      scale(al_a);
      fold8(0);
      if (doB) {
        scale(al_b);
        fold8(1);
      }
    } else {
      scale(al_a);
      fold(0);
      fold(1);
      if (doB) {
        scale(al_b);
        fold(2);
        fold(3);
      }
    }
  }

  __syncthreads();
#pragma unroll
  for (int n = 0; n < NQ; n++) {
    const float l = Ls[16 * n + c];
    // RN(acc / l) through one binary64 reciprocal, as in attn_fwd_bf16_kernel
    const double rl = otx_recip64(l);
    float x[4 * NT];  // output row r, tile j at X(r, j)
    auto X = [](int r, int j) { return I8 ? 4 * j + r : NT * r + j; };
    bool low = false;
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int j = 0; j < NT; j++) {
        x[X(r, j)] = otx_div_by_recip(acc[n][j][r], rl);
        low = low || !(__builtin_fabsf(x[X(r, j)]) >= 0x1p-126f);
      }
    if (__builtin_expect(__ballot(low) != 0, 0)) {
#pragma unroll
      for (int r = 0; r < 4; r++)
#pragma unroll
        for (int j = 0; j < NT; j++) x[X(r, j)] = otx_div_by_recip_checked(acc[n][j][r], rl, l);
    }
    T* dst = o + ((size_t)bh * S + q0 + 16 * n + c) * D + w * (D / 4);
    if constexpr (I8) {
#pragma unroll
      for (int j = 0; j < NT; j++) {
        const float y[4] = {x[4 * j], x[4 * j + 1], x[4 * j + 2], x[4 * j + 3]};
        tile_store(dst + 16 * j + 4 * g, y);
      }
    } else {
      tile_store(dst + NT * 4 * g, x);
    }
    if (w == 0 && g == n) lse[(size_t)bh * S + q0 + 16 * n + c] = m[n] + otx_logf_tile_call(l);
  }
}

// dK/dV.  A workgroup owns 16 NK consecutive keys of one KV head and walks the
// query blocks that see them (heads of the group outermost) in steps of 64 / NK
// queries, whose Q and dO rows it holds in LDS as binary32 (the next step's are
// in registers meanwhile):
//   wave (wq, wk): the 16 x 16 tiles of S and dP of queries 16 wq .. and keys
//        16 wk .. (A = Q, dO rows from LDS; B = K, V rows in registers), then
//        P and dS, which go to the other waves through LDS and, dS, to the dQ
//        kernel's tiles;
//   wave w: dV^T and dK^T of d = w D/4 .. for all the workgroup's keys (A = dO, Q
//        from LDS across rows; B = P, dS).
// Rows are D + 20 floats apart: the score reads (16 rows, four terms) then fall
// into 64 different banks and the fold reads (four rows, 16 columns) share a
// bank two at a time at most.  (D 128 with 64-query steps keeps D + 4, four at a
// time: then two workgroups fit a CU's LDS; 16 heads x 2048, nkb 1024, 428 -> 361
// us.)  8 heads, 2 KV heads x 1024 x 128, binary32: 1457 -> 222 us; 16 heads x 1024
// x 128, bf16 with the score cache: 118 -> 95 us.
template <typename T, int D, int NK, bool SC>
__global__ __launch_bounds__(256, 2) void attn_dkdv_tile_kernel(
    const T* __restrict__ q, const T* __restrict__ k, const T* __restrict__ v, const T* __restrict__ dO,
    const float* __restrict__ lse, const float* __restrict__ dsum, T* __restrict__ dk, T* __restrict__ dv,
    float* __restrict__ ws_ds, int B, int H, int Hkv, int S, int window, float sigma, int order,
    const float* __restrict__ scache) {
  constexpr int KS = D / 4;
  constexpr int NT = D / 64;
  constexpr int ROWS = 64 / NK;             // queries per step
  constexpr int NB = ROWS / OTX_BLK;        // query blocks per step
  constexpr int UPB = 2 / NK;               // workgroups per key block
  constexpr int RP = D + (NK == 1 && D == 128 ? 4 : 20);  // row pitch in floats
  constexpr int VEC = Elem<T>::VEC;
  constexpr int CH = D / VEC;               // 16-byte chunks of a row
  constexpr int NL = ROWS * CH / 256;       // chunks per thread and matrix
  __shared__ double tab[OTX_EXP_LE0_TAB_N];
  __shared__ __align__(16) float Qs[ROWS * RP];
  __shared__ __align__(16) float Gs[ROWS * RP];
  __shared__ float4 Xb[2][NK][ROWS / 16][64];
  __shared__ __align__(16) float Ll[ROWS], Dl[ROWS];

  const int nt = S / OTX_BLK, units = nt * UPB, BG = B * Hkv, G = H / Hkv;
  const int bid = blockIdx.x;
  int unit, bg;
  if (order == 0) {  // low keys are seen by the most queries: first
    unit = bid / BG;
    bg = bid % BG;
  } else {
    unit = units - 1 - bid % units;
    bg = bid / units;
  }
  const int b = bg / Hkv, g0 = bg % Hkv;
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), L = threadIdx.x & 63, g = L >> 4, c = L & 15;
  const int wq = NK == 2 ? w >> 1 : w, wk = NK == 2 ? w & 1 : 0;
  const int kt = unit / UPB, k0 = unit * 16 * NK;
  const int qhi = otx_qblock_hi(kt, window, nt);
  const int nsteps = (qhi - kt) / NB + 1;
  const long tiles_per_head = otx_tile_offset(nt, window);

  otx_load_exp_table(tab);
  float kr[SC ? 1 : KS], vr[KS];
  {
    const size_t off = ((size_t)bg * S + k0 + 16 * wk + c) * D + 4 * g;
#pragma unroll
    for (int u = 0; u < KS / 4; u++) {
      float a[4];
      if constexpr (!SC) {
        tile_get(tile_load<T, 4>(k + off + 16 * u), a);
        otx_transpose4(a);
#pragma unroll
        for (int e = 0; e < 4; e++) kr[4 * u + e] = a[e];
      }
      tile_get(tile_load<T, 4>(v + off + 16 * u), a);
      otx_transpose4(a);
#pragma unroll
      for (int e = 0; e < 4; e++) vr[4 * u + e] = a[e];
    }
  }

  uint4 qraw[NL], graw[NL];
  float lraw = 0.0f, draw = 0.0f;
  const int x0 = threadIdx.x;
  // chunk x of a step: row x / CH; a second block past the last is not used and loads the last one again
  static_assert(256 / CH <= OTX_BLK, "the chunks of one index lie in one block");
  auto load_step = [&](int r, int qb) {
    const size_t bh = (size_t)b * H + g0 * G + r;
    const size_t row0 = bh * S + (size_t)qb * OTX_BLK;
    const int back = NB == 2 && qb + 1 > qhi ? OTX_BLK : 0;
    const uint4* qp = reinterpret_cast<const uint4*>(q + row0 * D);
    const uint4* gp = reinterpret_cast<const uint4*>(dO + row0 * D);
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int x = x0 + 256 * i - (256 * i / CH >= OTX_BLK ? back * CH : 0);
      qraw[i] = qp[x];
      graw[i] = gp[x];
    }
    if (x0 < ROWS) {
      const size_t row = row0 + x0 - (x0 >= OTX_BLK ? back : 0);
      lraw = lse[row];
      draw = dsum[row];
    }
  };
  load_step(0, kt);

  f32x4 accV[NK][NT], accK[NK][NT];
#pragma unroll
  for (int n = 0; n < NK; n++)
#pragma unroll
    for (int j = 0; j < NT; j++) { accV[n][j] = f32x4{}; accK[n][j] = f32x4{}; }

  int r = 0, qb = kt;
  const int total = G * nsteps;
  for (int it = 0; it < total; ++it) {
    const size_t bh = (size_t)b * H + g0 * G + r;
#pragma unroll
    for (int i = 0; i < NL; i++) {
      const int x = x0 + 256 * i, off = (x / CH) * RP + (x % CH) * VEC;
#pragma unroll
      for (int e = 0; e < VEC; e += 4) {
        *reinterpret_cast<float4*>(Qs + off + e) =
            make_float4(Elem<T>::get(qraw[i], e), Elem<T>::get(qraw[i], e + 1), Elem<T>::get(qraw[i], e + 2),
                        Elem<T>::get(qraw[i], e + 3));
        *reinterpret_cast<float4*>(Gs + off + e) =
            make_float4(Elem<T>::get(graw[i], e), Elem<T>::get(graw[i], e + 1), Elem<T>::get(graw[i], e + 2),
                        Elem<T>::get(graw[i], e + 3));
      }
    }
    if (x0 < ROWS) {
      Ll[x0] = lraw;
      Dl[x0] = draw;
    }
    __syncthreads();
    const int qnow = qb;
    qb += NB;
    if (qb > qhi) {
      qb = kt;
      r++;
    }
    load_step(r < G ? r : G - 1, qb);

    const int qblk = qnow + (16 * wq) / OTX_BLK;
    if (qblk <= qhi) {  // always, but for the second block of a 64-query step past the end
      const long tile = (long)bh * tiles_per_head + otx_tile_offset(qblk, window) + (kt - otx_kblock_lo(qblk, window));
      const int qs = (16 * wq) & 31, ks = (k0 + 16 * wk) & 31;  // this wave's corner of the 32 x 32 tile
      float ex[4];
      f32x4 sa = f32x4{}, pa = f32x4{};
      const float* qrow = Qs + (16 * wq + c) * RP + g;
      const float* grow = Gs + (16 * wq + c) * RP + g;
      float4 sc4;
      if constexpr (SC) sc4 = *reinterpret_cast<const float4*>(scache + (tile << 10) + (ks + c) * 32 + qs + 4 * g);
#pragma unroll
      for (int t = 0; t < KS; t++) {
        if constexpr (!SC) sa = otx_mfma_k4(qrow[4 * t], kr[t], sa);
        pa = otx_mfma_k4(grow[4 * t], vr[t], pa);
      }
      const float4 l4 = *reinterpret_cast<const float4*>(Ll + 16 * wq + 4 * g);
      const float4 d4 = *reinterpret_cast<const float4*>(Dl + 16 * wq + 4 * g);
      float lv[4], dd[4];
      tile_get(l4, lv);
      tile_get(d4, dd);
      if constexpr (SC) {
        tile_get(sc4, ex);
      } else {
#pragma unroll
        for (int i = 0; i < 4; i++) ex[i] = sa[i] * sigma;
      }
      const bool need_mask = qblk == kt || (window > 0 && qblk == kt + window / OTX_BLK);
#pragma unroll
      for (int i = 0; i < 4; i++) {
        ex[i] = ex[i] - lv[i];
        if (need_mask)
          ex[i] = otx_masked(qblk * OTX_BLK + qs + 4 * g + i, k0 + 16 * wk + c, window) ? -__builtin_inff() : ex[i];
      }
      otx_exp_n<4, true, 4>(ex, tab);
      float* tds = ws_ds + (tile << 10) + (qs + 4 * g) * 32 + ks + c;
#pragma unroll
      for (int i = 0; i < 4; i++) {
        const float ds = ex[i] * (pa[i] - dd[i]);
        reinterpret_cast<float*>(&Xb[0][wk][wq][16 * i + c])[g] = ex[i];
        reinterpret_cast<float*>(&Xb[1][wk][wq][16 * i + c])[g] = ds;
        tds[32 * i] = ds;
      }
    }
    __syncthreads();
    const float* qcol = Qs + g * RP + w * (D / 4) + c;
    const float* gcol = Gs + g * RP + w * (D / 4) + c;
#pragma unroll
    for (int t4 = 0; t4 < ROWS / 16; t4++) {
      if (NB == 2 && t4 == 2 && qnow + 1 > qhi) break;
      float p[NK][4], ds[NK][4];
#pragma unroll
      for (int n = 0; n < NK; n++) {
        tile_get(Xb[0][n][t4][L], p[n]);
        tile_get(Xb[1][n][t4][L], ds[n]);
      }
#pragma unroll
      for (int e = 0; e < 4; e++)
#pragma unroll
        for (int j = 0; j < NT; j++) {
          const float ga = gcol[4 * (4 * t4 + e) * RP + 16 * j], qa = qcol[4 * (4 * t4 + e) * RP + 16 * j];
#pragma unroll
          for (int n = 0; n < NK; n++) {
            accV[n][j] = otx_mfma_k4(ga, p[n][e], accV[n][j]);
            accK[n][j] = otx_mfma_k4(qa, ds[n][e], accK[n][j]);
          }
        }
    }
    __syncthreads();
  }

#pragma unroll
  for (int n = 0; n < NK; n++)
#pragma unroll
    for (int j = 0; j < NT; j++) {
      const size_t off = ((size_t)bg * S + k0 + 16 * n + c) * D + w * (D / 4) + 16 * j + 4 * g;
      float x[4], y[4];
#pragma unroll
      for (int i = 0; i < 4; i++) {
        x[i] = accV[n][j][i];
        y[i] = accK[n][j][i] * sigma;
      }
      tile_store(dv + off, x);
      tile_store(dk + off, y);
    }
}

// dQ.  A workgroup owns 16 NQ consecutive queries of one head, wave w the
// columns d = w D/4 ..: no LDS and no barrier, K and the dS tiles come straight
// from global memory one key block ahead.  Beside the products its time is those
// loads (a K row per 32 queries and wave).  16 heads x 1024 x 128, bf16: 69 -> 30 us.
template <typename T, int D, int NQ>
__global__ __launch_bounds__(256, 2) void attn_dq_tile_kernel(const T* __restrict__ k,
                                                              const float* __restrict__ ws_ds, T* __restrict__ dq,
                                                              int B, int H, int Hkv, int S, int window, float sigma,
                                                              int order) {
  constexpr int NT = D / 64;
  constexpr int UPB = 2 / NQ;
  const int nqt = S / OTX_BLK, units = nqt * UPB, BH = B * H;
  const int bid = blockIdx.x;
  int unit, bh;
  if (order == 0) {
    unit = units - 1 - bid / BH;
    bh = bid % BH;
  } else {
    unit = bid % units;
    bh = bid / units;
  }
  const int b = bh / H, h = bh % H, gk = h / (H / Hkv);
  const int w = __builtin_amdgcn_readfirstlane(threadIdx.x >> 6), L = threadIdx.x & 63, g = L >> 4, c = L & 15;
  const int qt = unit / UPB, q0 = unit * 16 * NQ;
  const int lo = otx_kblock_lo(qt, window);
  const T* ksrc = k + (((size_t)b * Hkv + gk) * S + (size_t)lo * OTX_BLK + g) * D + w * (D / 4) + NT * c;
  const float* dsrc = ws_ds +
                      (((long)bh * otx_tile_offset(nqt, window) + otx_tile_offset(qt, window)) << 10) +
                      ((q0 & 31) + c) * 32 + 4 * g;
  typedef typename TileRaw<T, NT>::V RN;
  RN k0[8], k1[8];
  float4 d0[NQ][2], d1[NQ][2];
  auto load = [&](int i, RN (&kn)[8], float4 (&dn)[NQ][2]) {
    const T* kp = ksrc + (size_t)i * OTX_BLK * D;
    const float* dp = dsrc + ((long)i << 10);
#pragma unroll
    for (int n = 0; n < NQ; n++)
#pragma unroll
      for (int u = 0; u < 2; u++) dn[n][u] = *reinterpret_cast<const float4*>(dp + 512 * n + 16 * u);
#pragma unroll
    for (int t = 0; t < 8; t++) kn[t] = tile_load<T, NT>(kp + (size_t)4 * t * D);
  };
  f32x4 acc[NQ][NT];
#pragma unroll
  for (int n = 0; n < NQ; n++)
#pragma unroll
    for (int j = 0; j < NT; j++) acc[n][j] = f32x4{};
  load(0, k0, d0);
  const int nb = qt - lo;
  auto fold = [&](const RN (&kc)[8], const float4 (&dc)[NQ][2]) {
#pragma unroll
    for (int u = 0; u < 2; u++) {
      float ds[NQ][4];
#pragma unroll
      for (int n = 0; n < NQ; n++) {
        tile_get(dc[n][u], ds[n]);
        otx_transpose4(ds[n]);
      }
#pragma unroll
      for (int e = 0; e < 4; e++) {
        float x[NT];
        tile_get(kc[4 * u + e], x);
#pragma unroll
        for (int j = 0; j < NT; j++)
#pragma unroll
          for (int n = 0; n < NQ; n++) acc[n][j] = otx_mfma_k4(x[j], ds[n][e], acc[n][j]);
      }
    }
  };
  for (int i = 0; i <= nb; i += 2) {
    load(i + 1 < nb ? i + 1 : nb, k1, d1);
    __builtin_amdgcn_sched_barrier(0);  // the loads go out before this block's products
    fold(k0, d0);
    if (i == nb) break;
    load(i + 2 < nb ? i + 2 : nb, k0, d0);
    __builtin_amdgcn_sched_barrier(0);
    fold(k1, d1);
  }
#pragma unroll
  for (int n = 0; n < NQ; n++) {
    float x[4 * NT];
#pragma unroll
    for (int r = 0; r < 4; r++)
#pragma unroll
      for (int j = 0; j < NT; j++) x[NT * r + j] = acc[n][j][r] * sigma;
    tile_store(dq + ((size_t)bh * S + q0 + 16 * n + c) * D + w * (D / 4) + NT * 4 * g, x);
  }
}

// A launch holds fewer than 2^32 threads along x. binary32 forwards have no other kernel, and a card's memory holds
// more workgroups than that (2^23 blocks of 32 rows, D 64, two workgroups each: 69 GB of Q): they go along y too.
static dim3 fwd_tile_grid(long wgs) {
  constexpr long most = (1L << 24) - 1;
  const long y = (wgs + most - 1) / most;
  return dim3((unsigned)((wgs + y - 1) / y), (unsigned)y);
}

template <typename T, int D>
static hipError_t launch_fwd_tile_d(int nq, const void* q, const void* k, const void* v, void* o, float* lse, int B,
                                    int H, int Hkv, int S, int window, float sigma, int order, float* scache,
                                    hipStream_t st) {
  const dim3 grid = fwd_tile_grid((long)(S / OTX_BLK) * (2 / nq) * B * H);
#define OTX_FWD_TILE(NQ)                                                                                        \
  hipLaunchKernelGGL((attn_fwd_tile_kernel<T, D, NQ>), grid, dim3(256), 0, st, (const T*)q, (const T*)k, \
                     (const T*)v, (T*)o, lse, B, H, Hkv, S, window, sigma, order, scache, nullptr, nullptr)
  if (nq == 1) OTX_FWD_TILE(1); else OTX_FWD_TILE(2);
#undef OTX_FWD_TILE
  return hipGetLastError();
}

// int8-PV on the quantized V of attn_quant_v_kernel (qvt, vstep).
template <int D>
static hipError_t launch_fwd_tile_i8_d(int nq, const void* q, const void* k, void* o, float* lse, int B, int H, int Hkv,
                                       int S, int window, float sigma, int order, const int8_t* qvt,
                                       const float* vstep, float* scache, hipStream_t st) {
  const dim3 grid = fwd_tile_grid((long)(S / OTX_BLK) * (2 / nq) * B * H);
#define OTX_FWD_TILE(NQ)                                                                                    \
  hipLaunchKernelGGL((attn_fwd_tile_kernel<uint16_t, D, NQ, true>), grid, dim3(256), 0, st,           \
                     (const uint16_t*)q, (const uint16_t*)k, nullptr, (uint16_t*)o, lse, B, H, Hkv, S, window, \
                     sigma, order, scache, qvt, vstep)
  if (nq == 1) OTX_FWD_TILE(1); else OTX_FWD_TILE(2);
#undef OTX_FWD_TILE
  return hipGetLastError();
}

template <typename T, int D>
static hipError_t launch_dkdv_tile_d(int nk, const void* q, const void* k, const void* v, const void* dO,
                                     const float* lse, const float* dsum, void* dk, void* dv, float* ds, int B, int H,
                                     int Hkv, int S, int window, float sigma, int order, const float* scache,
                                     hipStream_t st) {
  const unsigned grid = (unsigned)((long)(S / OTX_BLK) * (2 / nk) * B * Hkv);
#define OTX_DKDV_TILE(NK, SC)                                                                                     \
  hipLaunchKernelGGL((attn_dkdv_tile_kernel<T, D, NK, SC>), dim3(grid), dim3(256), 0, st, (const T*)q,            \
                     (const T*)k, (const T*)v, (const T*)dO, lse, dsum, (T*)dk, (T*)dv, ds, B, H, Hkv, S, window, \
                     sigma, order, scache)
  if constexpr (sizeof(T) == 2) {
    if (scache != nullptr) {
      if (nk == 1) OTX_DKDV_TILE(1, true); else OTX_DKDV_TILE(2, true);
      return hipGetLastError();
    }
  } else if (scache != nullptr) {
    return hipErrorInvalidValue;  // the score cache is a bf16-path feature
  }
  if (nk == 1) OTX_DKDV_TILE(1, false); else OTX_DKDV_TILE(2, false);
#undef OTX_DKDV_TILE
  return hipGetLastError();
}

template <typename T, int D>
static hipError_t launch_dq_tile_d(int nq, const void* k, const float* ds, void* dq, int B, int H, int Hkv, int S,
                                   int window, float sigma, int order, hipStream_t st) {
  const unsigned grid = (unsigned)((long)(S / OTX_BLK) * (2 / nq) * B * H);
#define OTX_DQ_TILE(NQ)                                                                                          \
  hipLaunchKernelGGL((attn_dq_tile_kernel<T, D, NQ>), dim3(grid), dim3(256), 0, st, (const T*)k, ds, (T*)dq, B, \
                     H, Hkv, S, window, sigma, order)
  if (nq == 1) OTX_DQ_TILE(1); else OTX_DQ_TILE(2);
#undef OTX_DQ_TILE
  return hipGetLastError();
}

// dtype 1: bf16, otherwise binary32; n16: 16-row tiles per workgroup (1 or 2).
#define OTX_TILE_DISPATCH(FN, ...)                                                       \
  (dtype == 1 ? (D == 128 ? FN<uint16_t, 128>(__VA_ARGS__) : FN<uint16_t, 64>(__VA_ARGS__)) \
              : (D == 128 ? FN<float, 128>(__VA_ARGS__) : FN<float, 64>(__VA_ARGS__)))
hipError_t launch_fwd_tile(int dtype, int D, int n16, const void* q, const void* k, const void* v, void* o, float* lse,
                           int B, int H, int Hkv, int S, int window, float sigma, int order, float* scache,
                           hipStream_t st) {
  return OTX_TILE_DISPATCH(launch_fwd_tile_d, n16, q, k, v, o, lse, B, H, Hkv, S, window, sigma, order, scache, st);
}
hipError_t launch_fwd_tile_i8(int D, int n16, const void* q, const void* k, void* o, float* lse, int B, int H, int Hkv,
                              int S, int window, float sigma, int order, const int8_t* qvt, const float* vstep,
                              float* scache, hipStream_t st) {
  if (D == 128)
    return launch_fwd_tile_i8_d<128>(n16, q, k, o, lse, B, H, Hkv, S, window, sigma, order, qvt, vstep, scache, st);
  return launch_fwd_tile_i8_d<64>(n16, q, k, o, lse, B, H, Hkv, S, window, sigma, order, qvt, vstep, scache, st);
}
hipError_t launch_dkdv_tile(int dtype, int D, int n16, const void* q, const void* k, const void* v, const void* dO,
                            const float* lse, const float* dsum, void* dk, void* dv, float* ds, int B, int H, int Hkv,
                            int S, int window, float sigma, int order, const float* scache, hipStream_t st) {
  return OTX_TILE_DISPATCH(launch_dkdv_tile_d, n16, q, k, v, dO, lse, dsum, dk, dv, ds, B, H, Hkv, S, window, sigma,
                           order, scache, st);
}
hipError_t launch_dq_tile(int dtype, int D, int n16, const void* k, const float* ds, void* dq, int B, int H, int Hkv,
                          int S, int window, float sigma, int order, hipStream_t st) {
  return OTX_TILE_DISPATCH(launch_dq_tile_d, n16, k, ds, dq, B, H, Hkv, S, window, sigma, order, st);
}

}  // namespace otx
