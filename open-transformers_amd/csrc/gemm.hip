// bf16 GEMM with a serial binary32 fold, for the projections around the
// attention (Q/K/V/O, SwiGLU gate/up/down) and their backward.
//
// Replaces repop.nn.linear.Linear (src/pretrain/model/modules/_linear.py:31-65
// of the reference; bf16 operands, fp32 accumulate, bf16 result:
// docs/MODEL_OP_DTYPE_TRACE.md:82,100,165-167).  Contract:
//   C[i][j] = RN_out( acc ),  acc = +0; for r = 0 .. R-1 ascending:
//             acc = fma(A(i, r), B(j, r), acc)
// with A(i, r) = A[i*a_i + r*a_r] and B(j, r) = B[j*b_j + r*b_r] (element
// strides), bf16 values, RN_out = round-to-nearest-even bf16 (or none for a
// binary32 output).  bf16 x bf16 products are exact in binary32, so every
// step is one rounded addition and the order is the whole contract
// (docs/unified-audit-results.md:71-74: "strict sequential ... fold ... no
// split-K").  Each fma is one lane of a v_mfma_f32_32x32x1_2b_f32, whose
// chain over r is that serial fold.
//
// Tiling: a workgroup of 4 waves owns a 128 x 128 block of C, each wave a
// 64 x 64 quarter (two MFMAs per r: i-blocks {0,1} x j-block 0, then x
// j-block 1), or, in the narrow form (both operands i-contiguous), a 128 x 64 block
// with 64 x 32 per wave (one MFMA per r), or, in the small forms, a 64 x 64 or 32 x 32 block with
// 32 x 32 or 16 x 16 per wave, on v_mfma_f32_16x16x4_f32 (four serial fmas per
// output; see there).  The wide and narrow forms (gemm_bf16_v2_kernel)
// advance r in chunks of 32 kept in LDS as bf16 in two slots, one barrier per chunk:
// an i-contiguous operand is copied straight from global memory into LDS, an
// r-contiguous one loaded into registers and stored transposed, and the MFMA
// operands are read with ds_read_u16_d16_hi, which yields the binary32 value of
// a bf16 with no conversion instruction (see GemmTile16).  Either operand may be
// r-contiguous (a_r == 1) or i-contiguous (a_i == 1); the loads are 16-byte
// vectors along the contiguous axis.  Every output is one lane's serial chain
// whatever the tile, so every form gives the same bytes.
#include "otx_common.h"

namespace otx {

constexpr int GT = 128;   // workgroup tile (i and j)
constexpr int GRC = 32;   // r chunk

// Tile of workgroup `bid` among ntiles = tiles_i x tiles_j.  Workgroups are
// dealt to the 8 XCDs round-robin (workgroup b runs on XCD b % 8, each XCD with
// its own L2), so the tiles are renumbered to give every XCD a contiguous band,
// walked in groups of GM tile rows with the rows fastest: the workgroups that
// an XCD runs at once then share their A rows and B columns in its L2.  For the
// lm-head logits (64 x 1002 tiles) the B operand (the 128256-row weight, larger
// than the last-level cache) is streamed from HBM once per XCD instead of once
// per tile row: -4 %.  Any order gives the same bytes.
__device__ __forceinline__ void gemm_tile(int bid, int ntiles, int tiles_j, int* ti, int* tj) {
  constexpr int GM = 4;
  int s = bid;
  if ((ntiles & 7) == 0) s = (bid & 7) * (ntiles >> 3) + (bid >> 3);
  const int tiles_i = ntiles / tiles_j;
  const int first = (s / (GM * tiles_j)) * GM;
  const int gm = tiles_i - first < GM ? tiles_i - first : GM;
  const int within = s - first * tiles_j;
  *ti = first + within % gm;
  *tj = within / gm;
}

// One operand's chunk of 32 r held in LDS as bf16, [r][row] with a pitch of PB
// bytes per r, read by ds_read_u16_d16_hi straight into the binary32 operand
// registers (no conversion instruction).  An i-contiguous operand is copied
// straight from global memory (global_load_lds_dwordx4: each r row of the chunk
// is ROWS contiguous bf16, 1 KB per instruction); an r-contiguous one is loaded
// into registers (8 consecutive r of one row per 16-byte load) and written
// transposed with 2-byte stores, its pitch padded by 8 bytes so that the four r
// rows a wave writes at once fall in distinct banks.
template <bool RCONT, int ROWS>
struct GemmTile16 {
  static constexpr int PB = RCONT ? ROWS * 2 + 8 : ROWS * 2;
  static constexpr int BYTES = GRC * PB;
  static constexpr int NV = ROWS * GRC / 8 / 256;  // 16-byte loads per thread (r-contiguous)
  static constexpr int RPI = 1024 / (ROWS * 2);    // r rows per direct copy instruction
  static constexpr int NI = GRC / RPI / 4;         // direct copy instructions per wave
  static_assert(NV >= 1 && NI >= 1, "tile shape");
  uint4 v[RCONT ? NV : 1];
  __device__ __forceinline__ void issue(const uint16_t* base, long s_i, long s_r, int i0, int r0, unsigned char* slot,
                                        int wave_u, int L) {
    if constexpr (RCONT) {
#pragma unroll
      for (int x = 0; x < NV; x++) {
        const int idx = threadIdx.x + 256 * x;
        const int i = idx >> 2, rv = (idx & 3) * 8;
        v[x] = *reinterpret_cast<const uint4*>(base + (long)(i0 + i) * s_i + (r0 + rv));
      }
    } else {
#pragma unroll
      for (int x = 0; x < NI; x++) {
        const int rb = (wave_u + 4 * x) * RPI;
        const int r = rb + L / (ROWS / 8), iv = (L % (ROWS / 8)) * 8;
        otx_dma16(base + (long)(r0 + r) * s_r + (i0 + iv), slot + rb * PB);
      }
    }
  }
  __device__ __forceinline__ void commit(unsigned char* slot) const {
    if constexpr (RCONT) {
#pragma unroll
      for (int x = 0; x < NV; x++) {
        const int idx = threadIdx.x + 256 * x;
        const int i = idx >> 2, rv = (idx & 3) * 8;
        unsigned char* p = slot + rv * PB + i * 2;
        const uint32_t* w = reinterpret_cast<const uint32_t*>(&v[x]);
#pragma unroll
        for (int k = 0; k < 4; k++) {
          *reinterpret_cast<uint16_t*>(p + (2 * k) * PB) = (uint16_t)w[k];
          *reinterpret_cast<uint16_t*>(p + (2 * k + 1) * PB) = (uint16_t)(w[k] >> 16);
        }
      }
    }
  }
};

template <int N>
__device__ __forceinline__ void gemm_lds_wait6(float (&r)[6]) {
  asm volatile("s_waitcnt lgkmcnt(%6)"
               : "+v"(r[0]), "+v"(r[1]), "+v"(r[2]), "+v"(r[3]), "+v"(r[4]), "+v"(r[5])
               : "i"(N));
}

// The wide and narrow forms with bf16 LDS tiles, two slots and one barrier per
// chunk: chunk ch is read from slot ch & 1 while the copies of chunk ch + 1
// (issued one chunk earlier) land in the other slot.  The operands are read one
// group of two r ahead with hand-kept lgkmcnt accounting (six or four reads per
// group, at most twelve outstanding); the accumulators stay in the
// accumulation registers, so 64 vector registers remain and four workgroups
// share a CU (launch bound: four waves per SIMD).  No vector instruction
// converts or stages an i-contiguous operand, and an r-contiguous one costs
// only its 2-byte stores.
template <bool ARC, bool BRC, bool OUT_F32, int WJ>
__global__ __launch_bounds__(256, 4) void gemm_bf16_v2_kernel(const uint16_t* __restrict__ A, long a_i, long a_r,
                                                               const uint16_t* __restrict__ B, long b_j, long b_r,
                                                               void* __restrict__ C, long ldc, int M, int N, int R) {
  constexpr int GTJ = 2 * WJ;
  using TA = GemmTile16<ARC, GT>;
  using TB = GemmTile16<BRC, GTJ>;
  constexpr int SLOT = TA::BYTES + TB::BYTES;
  __shared__ __align__(16) unsigned char smem[2 * SLOT];
  const int tiles_j = N / GTJ;
  int ti, tj;
  gemm_tile(blockIdx.x, (M / GT) * tiles_j, tiles_j, &ti, &tj);
  const int i0 = ti * GT, j0 = tj * GTJ;
  const int wave = threadIdx.x >> 6, L = threadIdx.x & 63, hh = L >> 5, c = L & 31;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wi = (wave >> 1) * 64, wj = (wave & 1) * WJ;
  constexpr int NRD = WJ == 64 ? 6 : 4;  // reads per group of two r
  TA ta;
  TB tb;
  f32x32 acc0 = f32x32{}, acc1 = f32x32{};
  const int nch = R / GRC;
  auto slot_a = [&](int s) { return smem + s * SLOT; };
  auto slot_b = [&](int s) { return smem + s * SLOT + TA::BYTES; };
  ta.issue(A, a_i, a_r, i0, 0, slot_a(0), wave_u, L);
  tb.issue(B, b_j, b_r, j0, 0, slot_b(0), wave_u, L);
  ta.commit(slot_a(0));
  tb.commit(slot_b(0));
  if (nch > 1) {
    ta.issue(A, a_i, a_r, i0, GRC, slot_a(1), wave_u, L);
    tb.issue(B, b_j, b_r, j0, GRC, slot_b(1), wave_u, L);
  }
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  __syncthreads();
  float opr[2][6] = {};
  for (int ch = 0; ch < nch; ++ch) {
    const int s = ch & 1;
    const uint32_t aA = otx_lds_addr(slot_a(s)) + (wi + hh * 32 + c) * 2;
    const uint32_t aB = otx_lds_addr(slot_b(s)) + (wj + c) * 2;
    auto rd = [&](auto gc) {
      constexpr int G = decltype(gc)::value, BK = G & 1;
      OtxUnroll<0, 2>::run([&](auto ec) {
        constexpr int E = decltype(ec)::value, RR = 2 * G + E;
        otx_lds_bf16<RR * TA::PB>(opr[BK][E], aA);
        otx_lds_bf16<RR * TB::PB>(opr[BK][2 + E], aB);
        if constexpr (WJ == 64) otx_lds_bf16<RR * TB::PB + 64>(opr[BK][4 + E], aB);
      });
    };
    rd(std::integral_constant<int, 0>{});
    OtxUnroll<0, GRC / 2>::run([&](auto gc) {
      constexpr int G = decltype(gc)::value, BK = G & 1;
      if constexpr (G + 1 < GRC / 2) {
        rd(std::integral_constant<int, G + 1>{});
        gemm_lds_wait6<NRD>(opr[BK]);
      } else {
        gemm_lds_wait6<0>(opr[BK]);
      }
      OtxUnroll<0, 2>::run([&](auto ec) {
        constexpr int E = decltype(ec)::value;
        acc0 = otx_mfma(opr[BK][E], opr[BK][2 + E], acc0);
        if constexpr (WJ == 64) acc1 = otx_mfma(opr[BK][E], opr[BK][4 + E], acc1);
      });
      // bank BK is consumed before it is read again
      if constexpr (WJ == 64)
        asm volatile("" : "+a"(acc0), "+a"(acc1));
      else
        asm volatile("" : "+a"(acc0));
    });
    if (ch + 1 < nch) {
      ta.commit(slot_a(s ^ 1));
      tb.commit(slot_b(s ^ 1));
    }
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");  // this thread's copies of chunk ch + 1 have landed
    __syncthreads();  // chunk ch + 1 is visible, and slot s is no longer read
    if (ch + 2 < nch) {
      ta.issue(A, a_i, a_r, i0, (ch + 2) * GRC, slot_a(s), wave_u, L);
      tb.issue(B, b_j, b_r, j0, (ch + 2) * GRC, slot_b(s), wave_u, L);
    }
  }
  // acc0: rows wi + blk*32 + R(r%16, hh), column wj + c; acc1: column wj + 32 + c.
#pragma unroll
  for (int r = 0; r < 32; r++) {
    const int i = i0 + wi + 32 * (r >> 4) + otx_row(r, hh);
    const long o0 = (long)i * ldc + j0 + wj + c;
    if constexpr (OUT_F32) {
      static_cast<float*>(C)[o0] = acc0[r];
      if constexpr (WJ == 64) static_cast<float*>(C)[o0 + 32] = acc1[r];
    } else {
      static_cast<uint16_t*>(C)[o0] = otx_f32_to_bf16(acc0[r]);
      if constexpr (WJ == 64) static_cast<uint16_t*>(C)[o0 + 32] = otx_f32_to_bf16(acc1[r]);
    }
  }
}

// ---- the small forms: v_mfma_f32_16x16x4_f32 ----
// One instruction is four steps of the fold: D = fma(a3, b3, fma(a2, b2, fma(a1, b1,
// fma(a0, b0, C)))), each rounded (tests/test_gpu_selftest.py compares it with fmaf), in
// 32 cycles.  Its rate is that of the K = 1 forms, but a 16 x 16 block advances one r in 8
// cycles where they take 32 (or 64): a product with few tiles is bound by the chain
// of one wave, so the smaller block per wave is worth its operand traffic.  Lane
// L = 16 g + c supplies A row c and B column c of the block at r = 4 s + g, step s; result
// register q of lane L holds row 4 g + q, column c.
//
// A workgroup of 4 waves owns a 32 NB x 32 NB tile of C, each wave NB x NB blocks.  r
// advances in stages of 32 SUBS, kept in LDS as bf16 and copied straight from global
// memory (global_load_lds_dwordx4) three stages ahead into four slots, one barrier per
// stage.  An i-contiguous operand lies as [r][row]; an r-contiguous one as SUBS
// sub-chunks of [row][32 r], the four 16-byte units of a row swizzled by row / 4, so that
// the 16 rows that a step reads fall in distinct banks.  Either way a step reads its
// operands with ds_read_u16_d16_hi (no conversion, and no commit through registers),
// two groups ahead under hand-kept lgkmcnt accounting; no read is in flight across a
// branch, where the compiler could copy its register.
template <bool RC, int ROWS, int SUBS>
struct GemmStage {
  static constexpr int SUB = 32 * ROWS * 2;      // bytes of 32 r
  static constexpr int BYTES = SUBS * SUB;
  static constexpr int NI = BYTES / 1024 / 4;    // copy instructions per wave
  static constexpr int NA = RC ? 4 : 1;          // lane addresses
  static_assert(NI >= 1, "stage shape");
  // The stage of r0 on; r past the end of the product (a last stage that is not whole) copy its
  // first 32 again and are not read.
  __device__ __forceinline__ static void issue(const uint16_t* base, long s_i, long s_r, int i0, int r0, int R,
                                               unsigned char* lds, int wave_u, int L) {
#pragma unroll
    for (int x = 0; x < NI; x++) {
      const int n = wave_u + 4 * x;
      if constexpr (RC) {
        const int sub = n / (ROWS / 16), row = n % (ROWS / 16) * 16 + (L >> 2);
        const int unit = (L & 3) ^ ((row >> 2) & 3);
        const int r = r0 + (r0 + 32 * sub < R ? 32 * sub : 0) + 8 * unit;
        otx_dma16(base + (long)(i0 + row) * s_i + r, lds + n * 1024);
      } else {
        constexpr int VPR = ROWS / 8;  // vectors per r
        const int k = n * (64 / VPR) + L / VPR;
        const int r = r0 + k < R ? r0 + k : r0 + (k & 31);
        otx_dma16(base + (long)r * s_r + (i0 + L % VPR * 8), lds + n * 1024);
      }
    }
  }
  // Lane addresses (row0: the wave's first row), and the offset of block b at step s from address which(s).
  __device__ __forceinline__ static void lanes(uint32_t lds, int row0, int g, int c, uint32_t (&a)[NA]) {
    if constexpr (RC) {
#pragma unroll
      for (int u = 0; u < 4; u++) a[u] = lds + (row0 + c) * 64 + ((u ^ ((c >> 2) & 3)) << 4) + 2 * g;
    } else {
      a[0] = lds + g * ROWS * 2 + (row0 + c) * 2;
    }
  }
  static constexpr int which(int s) { return RC ? (s & 7) >> 1 : 0; }
  static constexpr int off(int s, int b) {
    return RC ? (s >> 3) * SUB + b * 16 * 64 + (s & 1) * 8 : 4 * s * ROWS * 2 + b * 32;
  }
};

template <int N>
__device__ __forceinline__ void gemm_vm_wait() {
  asm volatile("s_waitcnt vmcnt(%0)" ::"i"(N) : "memory");
}

typedef float f32x4 __attribute__((ext_vector_type(4)));

// f(0), f(1), ... f(E - 1) as long as they are true; whether all were.
template <int B, int E>
struct OtxAll {
  template <class F>
  __device__ __forceinline__ static bool run(F&& f) {
    if constexpr (B < E) {
      if (!f(std::integral_constant<int, B>{})) return false;
      return OtxAll<B + 1, E>::run(f);
    }
    return true;
  }
};

template <bool ARC, bool BRC, bool OUT_F32, int NB>
__global__ __launch_bounds__(256, 2) void gemm_bf16_k4_kernel(const uint16_t* __restrict__ A, long a_i, long a_r,
                                                               const uint16_t* __restrict__ B, long b_j, long b_r,
                                                               void* __restrict__ C, long ldc, int M, int N, int R) {
  constexpr int GS = 32 * NB;
  constexpr int NS = 4, P = NS - 1;
  constexpr int SUBS = NB == 1 ? 4 : 2, SR = 32 * SUBS;  // r per stage
  constexpr int SPG = NB == 1 ? 2 : 1;      // steps per read group
  using TA = GemmStage<ARC, GS, SUBS>;
  using TB = GemmStage<BRC, GS, SUBS>;
  constexpr int SLOT = TA::BYTES + TB::BYTES;
  constexpr int NDMA = TA::NI + TB::NI;     // copy instructions of a stage and wave
  static_assert(NS * SLOT <= 65536, "slot offsets are 16-bit immediates");
  static_assert(2 * NB * SPG == 4, "read group of 4");
  __shared__ __align__(16) unsigned char smem[NS * SLOT];
  const int tiles_j = N / GS;
  int ti, tj;
  gemm_tile(blockIdx.x, (M / GS) * tiles_j, tiles_j, &ti, &tj);
  const int i0 = ti * GS, j0 = tj * GS;
  const int wave = threadIdx.x >> 6, L = threadIdx.x & 63, g = L >> 4, c = L & 15;
  const int wave_u = __builtin_amdgcn_readfirstlane(wave);
  const int wi = (wave >> 1) * 16 * NB, wj = (wave & 1) * 16 * NB;
  const int nst = (R + SR - 1) / SR;
  const auto issue = [&](int st, unsigned char* slot) {
    TA::issue(A, a_i, a_r, i0, SR * st, R, slot, wave_u, L);
    TB::issue(B, b_j, b_r, j0, SR * st, R, slot + TA::BYTES, wave_u, L);
  };
#pragma unroll
  for (int k = 0; k < P; k++)
    if (k < nst) issue(k, smem + k * SLOT);
  uint32_t la[TA::NA], lb[TB::NA];
  TA::lanes(otx_lds_addr(smem), wi, g, c, la);
  TB::lanes(otx_lds_addr(smem) + TA::BYTES, wj, g, c, lb);
  f32x4 acc[NB][NB];
#pragma unroll
  for (int x = 0; x < NB; x++)
#pragma unroll
    for (int y = 0; y < NB; y++) acc[x][y] = f32x4{};
  float opr[3][4];  // read banks, low halves zero
#pragma unroll
  for (int x = 0; x < 4; x++) { opr[0][x] = 0.0f; opr[1][x] = 0.0f; opr[2][x] = 0.0f; }
  // every scalar load of an argument has returned before the counted LDS reads begin (they share lgkmcnt)
  asm volatile("s_waitcnt lgkmcnt(0)" : "+s"(ldc), "+s"(C));

  // The steps of SN sub-chunks from byte OFF of the addresses on.
  const auto steps = [&](auto offc, auto subc, const uint32_t (&pa)[TA::NA], const uint32_t (&pb)[TB::NA]) {
    constexpr int OFF = decltype(offc)::value, NG = decltype(subc)::value * 8 / SPG;
    const auto rd = [&](auto gc) {
      constexpr int G = decltype(gc)::value, BK = G % 3;
      OtxUnroll<0, SPG>::run([&](auto ec) {
        constexpr int E = decltype(ec)::value, ST = G * SPG + E;
        OtxUnroll<0, NB>::run([&](auto xc) {
          constexpr int X = decltype(xc)::value;
          otx_lds_bf16<OFF + TA::off(ST, X)>(opr[BK][E * 2 * NB + X], pa[TA::which(ST)]);
          otx_lds_bf16<OFF + TB::off(ST, X)>(opr[BK][E * 2 * NB + NB + X], pb[TB::which(ST)]);
        });
      });
    };
    rd(std::integral_constant<int, 0>{});
    rd(std::integral_constant<int, 1>{});
    OtxUnroll<0, NG>::run([&](auto gc) {
      constexpr int G = decltype(gc)::value, BK = G % 3;
      if constexpr (G + 2 < NG) {
        rd(std::integral_constant<int, G + 2>{});
        otx_lds_wait<8>(opr[BK]);
      } else if constexpr (G + 1 < NG) {
        otx_lds_wait<4>(opr[BK]);
      } else {
        otx_lds_wait<0>(opr[BK]);
      }
      OtxUnroll<0, SPG>::run([&](auto ec) {
        constexpr int E = decltype(ec)::value;
#pragma unroll
        for (int x = 0; x < NB; x++)
#pragma unroll
          for (int y = 0; y < NB; y++)
            acc[x][y] = __builtin_amdgcn_mfma_f32_16x16x4f32(opr[BK][E * 2 * NB + x], opr[BK][E * 2 * NB + NB + y],
                                                             acc[x][y], 0, 0, 0);
      });
      // bank BK is consumed before it is read again
#pragma unroll
      for (int x = 0; x < NB; x++)
#pragma unroll
        for (int y = 0; y < NB; y++) asm volatile("" : "+v"(acc[x][y]));
    });
  };
  int st = 0;
  const auto stage = [&](auto sc) {
    constexpr int S = decltype(sc)::value;
    if (st == nst) return false;
    // stage st has landed for every wave (the copies of at most P - 1 later ones stay in
    // flight), and stage st - 1 is no longer read
    if (nst - st > 2) gemm_vm_wait<2 * NDMA>();
    else if (nst - st == 2) gemm_vm_wait<NDMA>();
    else gemm_vm_wait<0>();
    asm volatile("s_barrier" ::: "memory");
    if (st + P < nst) issue(st + P, smem + ((S + P) % NS) * SLOT);
    if (SR * st + SR <= R) {
      steps(std::integral_constant<int, S * SLOT>{}, std::integral_constant<int, SUBS>{}, la, lb);
      st++;
      return true;
    }
    // a last stage that is not whole: its sub-chunks one by one (R is a multiple of 32)
    uint32_t pa[TA::NA], pb[TB::NA];
    for (int sub = 0; SR * st + 32 * sub < R; sub++) {
#pragma unroll
      for (int u = 0; u < TA::NA; u++) pa[u] = la[u] + S * SLOT + sub * TA::SUB;
#pragma unroll
      for (int u = 0; u < TB::NA; u++) pb[u] = lb[u] + S * SLOT + sub * TB::SUB;
      steps(std::integral_constant<int, 0>{}, std::integral_constant<int, 1>{}, pa, pb);
    }
    return false;
  };
  while (OtxAll<0, NS>::run(stage)) {
  }
#pragma unroll
  for (int x = 0; x < NB; x++)
#pragma unroll
    for (int y = 0; y < NB; y++)
#pragma unroll
      for (int q = 0; q < 4; q++) {
        const long o = (long)(i0 + wi + 16 * x + 4 * g + q) * ldc + j0 + wj + 16 * y + c;
        if constexpr (OUT_F32)
          static_cast<float*>(C)[o] = acc[x][y][q];
        else
          static_cast<uint16_t*>(C)[o] = otx_f32_to_bf16(acc[x][y][q]);
      }
}

template <bool ARC, bool BRC, int WJ>
static hipError_t launch_gemm_w(const void* A, long a_i, long a_r, const void* B, long b_j, long b_r, void* C,
                                long ldc, int M, int N, int R, bool out_f32, hipStream_t st) {
  const dim3 grid((unsigned)((M / GT) * (N / (2 * WJ)))), block(256);
  if (out_f32)
    hipLaunchKernelGGL((gemm_bf16_v2_kernel<ARC, BRC, true, WJ>), grid, block, 0, st, (const uint16_t*)A, a_i, a_r,
                       (const uint16_t*)B, b_j, b_r, C, ldc, M, N, R);
  else
    hipLaunchKernelGGL((gemm_bf16_v2_kernel<ARC, BRC, false, WJ>), grid, block, 0, st, (const uint16_t*)A, a_i, a_r,
                       (const uint16_t*)B, b_j, b_r, C, ldc, M, N, R);
  return hipGetLastError();
}

template <bool ARC, bool BRC, int NB>
static hipError_t launch_gemm_k4(const void* A, long a_i, long a_r, const void* B, long b_j, long b_r, void* C,
                                 long ldc, int M, int N, int R, bool out_f32, hipStream_t st) {
  const dim3 grid((unsigned)((M / (32 * NB)) * (N / (32 * NB)))), block(256);
  if (out_f32)
    hipLaunchKernelGGL((gemm_bf16_k4_kernel<ARC, BRC, true, NB>), grid, block, 0, st, (const uint16_t*)A, a_i, a_r,
                       (const uint16_t*)B, b_j, b_r, C, ldc, M, N, R);
  else
    hipLaunchKernelGGL((gemm_bf16_k4_kernel<ARC, BRC, false, NB>), grid, block, 0, st, (const uint16_t*)A, a_i, a_r,
                       (const uint16_t*)B, b_j, b_r, C, ldc, M, N, R);
  return hipGetLastError();
}

// form: 0 wide (128 x 128), 1 narrow (128 x 64), 2 small (64 x 64), 3 smallest (32 x 32).
template <bool ARC, bool BRC>
static hipError_t launch_gemm_t(const void* A, long a_i, long a_r, const void* B, long b_j, long b_r, void* C,
                                long ldc, int M, int N, int R, bool out_f32, int form, hipStream_t st) {
  if (form == 3) return launch_gemm_k4<ARC, BRC, 1>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, st);
  if (form == 2) return launch_gemm_k4<ARC, BRC, 2>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, st);
  if constexpr (!ARC && !BRC)
    if (form == 1) return launch_gemm_w<ARC, BRC, 32>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, st);
  return launch_gemm_w<ARC, BRC, 64>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, st);
}

// Tile choice (every form gives the same bytes): the form whose busiest CU has the least to
// do.  With t tiles of 128 x 128 on n CUs that CU works through m = ceil(t / n) wide tiles,
// ceil(2t / n) narrow, ceil(4t / n) 64 x 64 or ceil(16t / n) 32 x 32 ones.  What a tile takes
// over its matrix instructions (fitted to products of R 512 to 8192 and 16 to 5632 tiles,
// 4 us of launch taken off) is, for m = 1, 2 and more:
//                        y = x w^T          dx = dy w          dw = dy^T x
//   wide               1.24 1.17 1.12     1.19 1.14 1.10     1.09 1.10 1.085
//   narrow            (1.43 1.26 1.16)   (1.40 1.27 1.18)    1.19 1.11 1.10
//   64 x 64            1.25 1.17 1.15     1.25 1.17 1.18     1.25 1.17 1.18
//   32 x 32            1.41 throughout
// (few waves per SIMD expose a wide tile's waits; an r-contiguous operand costs the wide and
// narrow forms their commits, where the small forms copy it as it is).  Measured, before
// and now: 256 x 512 over 2048 (the k projection of a short batch) 46.7 -> 13.8 us, 32 x 32
// tiles; 1024 x 1024 over 1024 27 -> 21 us and 1280 x 5632 over 2048 267 -> 229 us, 64 x 64;
// 8192 x 11264 over 2048 stays with the wide form's 2.71 ms.  The narrow form is left to
// products with both operands i-contiguous (11264 x 2048 over 8192, 5.5 wide tiles per CU:
// 2.66 ms against 2.84 and 2.86); elsewhere the 64 x 64 form was as fast or faster (the figures
// in brackets), and the narrow form is not built.
// variant 1, 2, 3 and 4 force the wide, the narrow (where it exists), the 64 x 64 and the
// 32 x 32 form.
static int gemm_form(int M, int N, bool arc, bool brc, int variant) {
  const int lay = arc && brc ? 0 : arc || brc ? 1 : 2;
  if (variant >= 1 && (variant != 2 || lay == 2)) return variant - 1;
  const long t = (long)(M / GT) * (N / GT), n = otx_cu_count();
  static const long wide[3][3] = {{1240, 1170, 1120}, {1190, 1140, 1100}, {1090, 1100, 1085}};
  static const long narrow[3] = {1190, 1110, 1100};
  static const long small[3][3] = {{1250, 1170, 1150}, {1250, 1170, 1180}, {1250, 1170, 1180}};
  long best = 1410 * ((16 * t + n - 1) / n);  // in 1/16000 of a wide tile's matrix instructions
  int form = 3;
  for (int f = 2; f >= 0; f--) {
    if (f == 1 && lay != 2) continue;
    const long* over = f == 2 ? small[lay] : f == 1 ? narrow : wide[lay];
    const long m = ((t << f) + n - 1) / n, cost = m * (16 >> f) * over[m < 3 ? m - 1 : 2];
    if (cost <= best) {
      best = cost;
      form = f;
    }
  }
  return form;
}

hipError_t launch_gemm(const void* A, long a_i, long a_r, const void* B, long b_j, long b_r, void* C, long ldc, int M,
                       int N, int R, bool out_f32, int variant, hipStream_t st) {
  const bool arc = a_r == 1, brc = b_r == 1;
  const int f = gemm_form(M, N, arc, brc, variant);
  if (arc && brc) return launch_gemm_t<true, true>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, f, st);
  if (arc) return launch_gemm_t<true, false>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, f, st);
  if (brc) return launch_gemm_t<false, true>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, f, st);
  return launch_gemm_t<false, false>(A, a_i, a_r, B, b_j, b_r, C, ldc, M, N, R, out_f32, f, st);
}

}  // namespace otx
