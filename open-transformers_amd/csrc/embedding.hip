// Token embedding with a deterministic backward, for gfx950.
//
// Replaces repop.nn.embedding.Embedding (_DeterministicEmbeddingFn), used by
// src/pretrain/model/modules/embedding_repop.py:33-40 of the reference:
// forward = plain gather of weight rows; backward = "stable-sort + fixed-order
// segment scatter-add", fp32 accumulation, result in the gradient's dtype
// (docs/MODEL_OP_DTYPE_TRACE.md:75,106).  Contract:
//   grad_w[v][d] = RN_dtype( fold over positions p ascending with ids[p] == v
//                            of g[p][d], serial binary32 additions from +0 )
//   rows of ids that do not occur are +0; ids outside [0, V) are skipped in the
//   backward and give NaN rows in the forward.
// Backward pipeline: a stable radix sort of the ids (an integer permutation;
// positions of equal ids stay ascending), in one workgroup's LDS up to 16384
// positions and with hipCUB beyond; then one launch whose first workgroups fold
// the segments (one per sorted index that starts a segment) and whose last ones
// write the rows of absent ids as zeros meanwhile.
#include <hipcub/hipcub.hpp>
#include "otx_common.h"

namespace otx {

template <typename T>
__global__ __launch_bounds__(256) void emb_fwd_kernel(const int64_t* __restrict__ ids, const T* __restrict__ w,
                                                      T* __restrict__ out, long npos, int V, int D) {
  const long p = blockIdx.x;
  const int d = (blockIdx.y * 256 + threadIdx.x) * (int)(16 / sizeof(T));
  if (p >= npos || d >= D) return;
  const long id = ids[p];
  uint4 val;
  if (id >= 0 && id < V) {
    val = *reinterpret_cast<const uint4*>(w + id * (long)D + d);
  } else {
    const uint32_t nan = sizeof(T) == 2 ? 0x7fc07fc0u : 0x7fc00000u;
    val = make_uint4(nan, nan, nan, nan);
  }
  *reinterpret_cast<uint4*>(out + p * (long)D + d) = val;
}

// keys = ids (V for ids outside [0, V)), values = positions
__global__ __launch_bounds__(256) void emb_keys_kernel(const int64_t* __restrict__ ids, int* __restrict__ keys,
                                                       int* __restrict__ pos, long npos, int V) {
  const long p = (long)blockIdx.x * 256 + threadIdx.x;
  if (p >= npos) return;
  const long id = ids[p];
  keys[p] = (id >= 0 && id < V) ? (int)id : V;
  pos[p] = (int)p;
}

// The whole sort in one workgroup: n <= 16384 words (id << 14 | position) in LDS,
// 6 bits of the id per pass.  A wave owns a contiguous run of the words, 64 at a
// time; a word's place is the number of words with smaller digits, plus those of
// its digit in earlier waves and rounds, plus the lanes before it with the same
// digit (six ballots), so the order is stable.  One launch and no temporary
// storage, where the device-wide sort takes six launches: at 8192 ids of a
// 128256-word vocabulary those took about 30 us.
constexpr int EMB_SORT_MAX = 16384, EMB_POS_BITS = 14, EMB_DIGIT = 6, EMB_BINS = 1 << EMB_DIGIT;
constexpr int EMB_SORT_T = 1024, EMB_SORT_W = EMB_SORT_T / 64, EMB_SORT_R = EMB_SORT_MAX / EMB_SORT_T;

__global__ __launch_bounds__(EMB_SORT_T) void emb_sort_kernel(const int64_t* __restrict__ ids,
                                                              int* __restrict__ skeys, int* __restrict__ spos, int n,
                                                              int V, int bits) {
  __shared__ uint32_t buf[2][EMB_SORT_MAX];
  __shared__ uint32_t hist[EMB_SORT_W][EMB_BINS];
  __shared__ uint32_t wsum[EMB_SORT_W];
  const int t = threadIdx.x, wave = t >> 6, L = t & 63;
  const int rounds = (n + EMB_SORT_T - 1) / EMB_SORT_T, run0 = wave * rounds * 64;
  for (int i = t; i < rounds * EMB_SORT_T; i += EMB_SORT_T) {
    uint32_t w = 0xffffffffu;  // past the end: sorts after every id, V (the invalid ids) included
    if (i < n) {
      const long id = ids[i];
      w = ((id >= 0 && id < V ? (uint32_t)id : (uint32_t)V) << EMB_POS_BITS) | (uint32_t)i;
    }
    buf[0][i] = w;
  }
  int src = 0;
  for (int sh = EMB_POS_BITS; sh < EMB_POS_BITS + bits; sh += EMB_DIGIT) {
    hist[wave][L] = 0;
    __syncthreads();
    uint32_t word[EMB_SORT_R], off[EMB_SORT_R];
#pragma unroll
    for (int r = 0; r < EMB_SORT_R; r++) {
      if (r >= rounds) break;
      word[r] = buf[src][run0 + 64 * r + L];
      const uint32_t d = (word[r] >> sh) & (EMB_BINS - 1);
      uint64_t same = ~0ull;
#pragma unroll
      for (int b = 0; b < EMB_DIGIT; b++) {
        const uint64_t bal = __ballot((d >> b) & 1);
        same &= ((d >> b) & 1) ? bal : ~bal;
      }
      const int before = __popcll(same & ((1ull << L) - 1));
      off[r] = hist[wave][d] + before;
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
      if (before == 0) hist[wave][d] += __popcll(same);
      __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
    }
    __syncthreads();
    // exclusive prefix over (digit, wave), digit-major: thread t holds digit t / 16, wave t % 16
    const uint32_t mine = hist[t % EMB_SORT_W][t / EMB_SORT_W];
    uint32_t sum = mine;
#pragma unroll
    for (int o = 1; o < 64; o <<= 1) {
      const uint32_t y = __shfl_up(sum, o);
      if (L >= o) sum += y;
    }
    if (L == 63) wsum[wave] = sum;
    __syncthreads();
    uint32_t base = 0;
    for (int w = 0; w < wave; w++) base += wsum[w];
    hist[t % EMB_SORT_W][t / EMB_SORT_W] = base + sum - mine;
    __syncthreads();
#pragma unroll
    for (int r = 0; r < EMB_SORT_R; r++) {
      if (r >= rounds) break;
      buf[src ^ 1][hist[wave][(word[r] >> sh) & (EMB_BINS - 1)] + off[r]] = word[r];
    }
    src ^= 1;
    __syncthreads();
  }
  for (int i = t; i < n; i += EMB_SORT_T) {
    skeys[i] = (int)(buf[src][i] >> EMB_POS_BITS);
    spos[i] = (int)(buf[src][i] & (EMB_SORT_MAX - 1));
  }
}

// First sorted index whose key is >= v (npos if none); every lane of a wave calls it.
__device__ __forceinline__ int emb_lower_bound(const int* __restrict__ skeys, int npos, int v) {
  int lo = 0, hi = npos;  // the answer lies in [lo, hi]
  while (lo < hi) {
    const int step = (hi - lo + 63) / 64, i = lo + (int)(threadIdx.x & 63) * step;
    const int below = __popcll(__ballot(i < hi && skeys[i] < v));  // a prefix of the probes
    if (below == 0) return lo;
    const int last = lo + (below - 1) * step;  // the last probe below v
    hi = last + step < hi ? last + step : hi;
    lo = last + 1;
  }
  return lo;
}

// 16 bytes of a gradient row; without VEC the row need not be aligned.
template <typename T, bool VEC>
__device__ __forceinline__ uint4 emb_load16(const T* p) {
  if constexpr (VEC) return *reinterpret_cast<const uint4*>(p);
  uint4 v;
  uint32_t* w = reinterpret_cast<uint32_t*>(&v);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if constexpr (sizeof(T) == 2)
      w[k] = (uint32_t)p[2 * k] | ((uint32_t)p[2 * k + 1] << 16);
    else
      w[k] = __float_as_uint(p[k]);
  }
  return v;
}

// Workgroups [0, nfold): if sorted index i starts a segment of a valid id, fold the
// segment's rows in position order, 16 bytes of columns per thread.  The adds of a
// column are a serial chain over the segment; the rows are loaded EMB_PF at a time,
// the next batch under the adds of the current one, so that a long segment (a
// frequent token) costs one memory latency per batch and not one per row.
// Workgroups [nfold, gridDim.x): zeros for the rows of absent ids, whole runs of
// rows each; they write while the long segments are folded.  At 8192 positions
// with frequencies falling as 1 / rank (483 rows in the longest segment) and a
// 128256 x 2048 bf16 table, bound by the 525 MB of the table: forward and backward
// 402 -> 165 us (the fold waited 0.5 us per row of the longest segment, 244 us,
// after a zero fill of the whole table, 96 us).
constexpr int EMB_PF = 16;
template <typename T, bool VEC>
__global__ __launch_bounds__(256) void emb_fold_kernel(const int* __restrict__ skeys, const int* __restrict__ spos,
                                                       const T* __restrict__ g, T* __restrict__ gw, int npos, int V,
                                                       int D, int nfold) {
  constexpr int N = 16 / sizeof(T);
  __shared__ int list[256];
  const int t = threadIdx.x;
  if ((int)blockIdx.x >= nfold) {
    if (blockIdx.y != 0) return;
    const int nz = (int)gridDim.x - nfold, per = (V + nz - 1) / nz, z = (int)blockIdx.x - nfold;
    const int vpr = D / N;
    const long end = (long)(z + 1) * per < V ? (long)(z + 1) * per : V;
    for (long v0 = (long)z * per; v0 < end; v0 += 256) {
      const int rows = end - v0 < 256 ? (int)(end - v0) : 256;
      list[t] = 0;
      __syncthreads();
      for (int i = emb_lower_bound(skeys, npos, (int)v0) + t; i < npos && skeys[i] < v0 + rows; i += 256)
        list[skeys[i] - v0] = 1;
      __syncthreads();
      uint4* dst = reinterpret_cast<uint4*>(gw + v0 * D);
      for (long e = t; e < (long)rows * vpr; e += 256)
        if (!list[(uint32_t)e / (uint32_t)vpr]) dst[e] = make_uint4(0u, 0u, 0u, 0u);
      __syncthreads();
    }
    return;
  }
  const int i = blockIdx.x;
  const int key = skeys[i];
  if (key >= V || (i > 0 && skeys[i - 1] == key)) return;
  const int d = (blockIdx.y * 256 + t) * N;
  const bool live = d < D;
  const T* col = g + (live ? d : 0);
  float acc[N];
#pragma unroll
  for (int e = 0; e < N; e++) acc[e] = 0.0f;
  for (int c0 = i;; c0 += 256) {
    const bool in = c0 + t < npos && skeys[c0 + t] == key;  // a prefix of the threads
    if (in) list[t] = spos[c0 + t];
    const int n = __syncthreads_count(in);
    uint4 nxt[EMB_PF];
    const auto issue = [&](int r0) {
#pragma unroll
      for (int k = 0; k < EMB_PF; k++)
        if (r0 + k < n) nxt[k] = emb_load16<T, VEC>(col + (long)list[r0 + k] * D);
    };
    issue(0);
    for (int r0 = 0; r0 < n; r0 += EMB_PF) {
      uint4 cur[EMB_PF];
#pragma unroll
      for (int k = 0; k < EMB_PF; k++) cur[k] = nxt[k];
      issue(r0 + EMB_PF);
#pragma unroll
      for (int k = 0; k < EMB_PF; k++)
        if (r0 + k < n)
#pragma unroll
          for (int e = 0; e < N; e++) acc[e] = acc[e] + Elem<T>::get(cur[k], e);
    }
    if (n < 256) break;
    __syncthreads();  // the list is rewritten
  }
  if (!live) return;
  uint4 out;
  uint32_t* w = reinterpret_cast<uint32_t*>(&out);
#pragma unroll
  for (int k = 0; k < 4; k++) {
    if constexpr (sizeof(T) == 2)
      w[k] = (uint32_t)Elem<T>::put(acc[2 * k]) | ((uint32_t)Elem<T>::put(acc[2 * k + 1]) << 16);
    else
      w[k] = __float_as_uint(acc[k]);
  }
  *reinterpret_cast<uint4*>(gw + (long)key * D + d) = out;
}

static int key_bits(int V) {
  int b = 1;
  while ((1L << b) <= V) b++;  // keys are 0..V
  return b;
}

// Whether one workgroup's LDS sort serves (the id and the position share a 32-bit word).
static bool emb_lds_sort(long npos, int V) {
  return npos <= EMB_SORT_MAX && key_bits(V) + EMB_POS_BITS <= 32;
}

// Temporary storage of the key sort (some even where the LDS sort needs none: 0
// says that the size query failed).
size_t emb_sort_temp_bytes(long npos, int V) {
  if (emb_lds_sort(npos, V)) return 256;
  size_t bytes = 0;
  const hipError_t e = hipcub::DeviceRadixSort::SortPairs(nullptr, bytes, (const int*)nullptr, (int*)nullptr,
                                                          (const int*)nullptr, (int*)nullptr, (int)npos, 0, key_bits(V));
  return e == hipSuccess ? bytes : 0;
}

hipError_t launch_emb_fwd(int dtype, const int64_t* ids, const void* w, void* out, long npos, int V, int D,
                          hipStream_t st) {
  const int per = dtype == 1 ? 8 : 4;
  const dim3 grid((unsigned)npos, (unsigned)((D / per + 255) / 256)), block(256);
  if (dtype == 1)
    hipLaunchKernelGGL((emb_fwd_kernel<uint16_t>), grid, block, 0, st, ids, (const uint16_t*)w, (uint16_t*)out, npos,
                       V, D);
  else
    hipLaunchKernelGGL((emb_fwd_kernel<float>), grid, block, 0, st, ids, (const float*)w, (float*)out, npos, V, D);
  return hipGetLastError();
}

// ws: keys, pos, sorted keys, sorted pos (npos int32 each, 256-byte aligned), then hipCUB temp storage.
hipError_t launch_emb_bwd(int dtype, const int64_t* ids, const void* g, void* gw, long npos, int V, int D, char* ws,
                          size_t temp_bytes, hipStream_t st) {
  const size_t arr = ((size_t)npos * 4 + 255) / 256 * 256;
  int* keys = (int*)ws;
  int* pos = (int*)(ws + arr);
  int* skeys = (int*)(ws + 2 * arr);
  int* spos = (int*)(ws + 3 * arr);
  void* temp = ws + 4 * arr;
  hipError_t e = hipSuccess;
  if (emb_lds_sort(npos, V)) {
    hipLaunchKernelGGL(emb_sort_kernel, dim3(1), dim3(EMB_SORT_T), 0, st, ids, skeys, spos, (int)npos, V,
                       key_bits(V));
    e = hipGetLastError();
  } else {
    hipLaunchKernelGGL(emb_keys_kernel, dim3((unsigned)((npos + 255) / 256)), dim3(256), 0, st, ids, keys, pos, npos,
                       V);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    e = hipcub::DeviceRadixSort::SortPairs(temp, temp_bytes, keys, skeys, pos, spos, (int)npos, 0, key_bits(V), st);
  }
  if (e != hipSuccess) return e;
  // zero-row workgroups: at least 8 rows each, up to eight workgroups per CU
  const long want = ((long)V + 7) / 8, most = 8L * otx_cu_count();
  const unsigned nz = (unsigned)(want < most ? want : most);
  const bool vec = ((uintptr_t)g & 15u) == 0;
  const dim3 block(256);
  const auto launch = [&](unsigned nfold, unsigned nzero) {
    const int per = dtype == 1 ? 8 : 4;
    const dim3 grid(nfold + nzero, nfold ? (unsigned)((D + 256 * per - 1) / (256 * per)) : 1u);
#define OTX_EMB_FOLD(T, VEC)                                                                                     \
  hipLaunchKernelGGL((emb_fold_kernel<T, VEC>), grid, block, 0, st, skeys, spos, (const T*)g, (T*)gw, (int)npos, V, \
                     D, (int)nfold)
    if (dtype == 1) {
      if (vec) OTX_EMB_FOLD(uint16_t, true); else OTX_EMB_FOLD(uint16_t, false);
    } else {
      if (vec) OTX_EMB_FOLD(float, true); else OTX_EMB_FOLD(float, false);
    }
#undef OTX_EMB_FOLD
  };
  // a launch holds fewer than 2^32 threads along x: with so many positions the zeros go in one of their own
  if ((npos + nz) * 256 < (1L << 32)) {
    launch((unsigned)npos, nz);
  } else {
    launch(0, nz);
    e = hipGetLastError();
    if (e != hipSuccess) return e;
    launch((unsigned)npos, 0);
  }
  return hipGetLastError();
}

}  // namespace otx
