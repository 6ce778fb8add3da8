// Dense fp8 1d1d GEMMs of few output tiles (source/glm_deepgemm.cu:17-24, 38-39; scripts/glm_ops.py:57-78): one
// output tile per workgroup through a deep LDS ring.
//
// What bounds them.  A GEMM of some rows streams its weights once and runs a serial chain of K blocks per tile: the
// sums keep the order of the other kernels (64 of K after 64 of K into one f32 accumulator, so the outputs are
// identical), K is never split, and the only parallelism is over output tiles.  With a ring of two stages a workgroup
// waits for a memory round trip per K block (0.9 us of a 128 x 128 x 128 block whose MFMAs take 0.2); here NS stages
// are in flight, and the tile shapes below let a GEMM of any size spread over the CUs in about one round.  What is
// left per block is the copy into LDS: a CU takes 86-103 GB/s of operands that sit in its L2 (tiles of 64 x 64 on) and
// 62-67 GB/s in a GEMM whose weights come from HBM, whatever the ring's depth, the number of waves or the path (VGPRs or
// LDS), so a block of 128 x 192 (40 KB) takes 0.61-0.68 us where its MFMAs take 0.32.  Weights from HBM, M x N x K, two-stage ring -> this one: 7 x 2752
// x 6144 43 -> 10.7 us, 150 x 20480 x 2048 25 -> 18, 420 x 6144 x 12288 88 -> 62, 1000 x 6144 x 16384 147 -> 97.
//
// Kernel.  NW waves, of which WM x WN compute: wave (wm, wn) owns TJ x TI MFMA tiles of 32 x 32 (v_mfma_scale
// 32x32x64, weights as the first operand, as in kg_fp8_gemm.hip); all NW waves copy.  A stage is KBS blocks of 128
// of K of both operands: 128-byte rows (swizzled as in kg_fp8_gemm.hip) moved by buffer_load ... lds, 1 KB (8 rows)
// per instruction, each block of BM activation rows and BN weight rows.  Stage s lives in buffer s % NS, each its
// own __shared__ array (the compiler then sees that a copy into one does not alias the reads of another).
//   * A stage is NT MFMA slots; after a slot come at most FR fragment reads and CPS copies (in bursts they keep the
//     matrix pipe waiting: 104 -> 97 us at 1000 x 6144 x 16384).  Fragments are read one unit (U of the stage's 2 KBS
//     halves of 64 of K) ahead of their MFMAs into one of two register sets; the first unit of stage s + 1 is read
//     during the last unit of stage s.
//   * One barrier per stage, after slot BAR: this wave's copies of stage s + 1 have landed (the (NS - 2) NQ younger
//     ones may still be in flight) and its reads of stage s are done; after it the copies of stage s + NS go into the
//     buffer of stage s, the first C1 before the stage's end and the others in the next stage's slots up to BAR.
//   * The scale words (four K blocks each) sit in a register ring of DW groups, reloaded DW groups ahead; the
//     MFMA picks its byte by op_sel.
#include "kg_device.h"
#include "kg_host.h"

#include "kg_fp8_common.h"
#include "kg_ring.h"

template <int WM, int WN, int TJ, int TI, int NW, int NS, int KBS, int U, int BOFF, int FR, int CPS>
struct KgRing {
  static constexpr int BM = WM * TJ * 32, BN = WN * TI * 32, BLK = (BM + BN) * 128, STAGE = BLK * KBS;
  static constexpr int THREADS = NW * 64;
  static constexpr int NQ = (BM + BN) / 8 * KBS / NW;      // copy instructions per wave and stage
  static constexpr int BODY = NS == 3 ? 12 : 8;            // stages per loop body: whole rings, whole words
  static constexpr int DW = BODY * KBS / 4;                // word groups per body
  static constexpr int H = 2 * KBS, UPS = H / U;           // K halves of a stage, units of it
  static constexpr int NT = H * TI * TJ;                   // MFMA slots of a stage
  static constexpr int BAR = (UPS - 1) * U * TI * TJ + BOFF;   // the slot after which the barrier sits
  static constexpr int C1 = NQ < (NT - 1 - BAR) * CPS ? NQ : (NT - 1 - BAR) * CPS;   // copies issued after it
  static_assert(BODY % NS == 0 && BODY * KBS % 4 == 0 && NW % 2 == 0 && NW >= WM * WN && UPS <= 2, "ring");
  static_assert((BM / 8) % NW == 0 && (BN / 8) % NW == 0 && BAR < NT - 1 && NQ - C1 <= BAR * CPS, "copy split");
  static_assert(NS * STAGE <= 160 * 1024 && (NS - 1) * NQ < 60, "LDS and vmcnt");
};

template <int WM, int WN, int TJ, int TI, int NW, int NS, int KBS, int U, int BOFF, int FR, int CPS>
__global__ __launch_bounds__(NW * 64) void kg_fp8_gemm_ring(const KgFp8Args p) {
  using R = KgRing<WM, WN, TJ, TI, NW, NS, KBS, U, BOFF, FR, CPS>;
  constexpr int BM = R::BM, BN = R::BN, BLK = R::BLK, STAGE = R::STAGE, NQ = R::NQ, BODY = R::BODY, DW = R::DW;
  constexpr int UPS = R::UPS, NT = R::NT, BAR = R::BAR, C1 = R::C1, QA = BM / 8 / NW, QB = BN / 8 / NW;
  constexpr int NF = U * (TI + TJ);                       // fragments of a unit
  __shared__ __attribute__((aligned(1024))) u8 st0[STAGE];
  __shared__ __attribute__((aligned(1024))) u8 st1[STAGE];
  __shared__ __attribute__((aligned(1024))) u8 st2[NS > 2 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) u8 st3[NS > 3 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) u8 st4[NS > 4 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) u8 st5[NS > 4 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) u8 st6[NS > 4 ? STAGE : 16];
  __shared__ __attribute__((aligned(1024))) u8 st7[NS > 4 ? STAGE : 16];
  auto buf = [&](auto i) __attribute__((always_inline)) -> u8* {
    constexpr int x = decltype(i)::value % NS;
    if constexpr (x == 0) return st0;
    else if constexpr (x == 1) return st1;
    else if constexpr (x == 2) return st2;
    else if constexpr (x == 3) return st3;
    else if constexpr (x == 4) return st4;
    else if constexpr (x == 5) return st5;
    else if constexpr (x == 6) return st6;
    else return st7;
  };

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave % WM, wn = wave / WM;

  // Tile order: groups of G = 8 row tiles, column-tile-major inside a group, a contiguous range per XCD, so that
  // the workgroups an XCD runs at once share row tiles and weight slices through its L2.
  constexpr int G = 8;
  const int wid = kg_xcd_remap((int)blockIdx.x, (int)gridDim.x);
  const int gsz = G * p.n_tiles, grp = wid / gsz, first = grp * G;
  const int gm = min(p.m_tiles - first, G), r = wid - grp * gsz;
  const int m0 = (first + r % gm) * BM, m_end = min(p.m, m0 + BM), n0 = r / gm * BN;
  const int kw = (p.k + 511) >> 9, KB = p.k >> 7, KS = (KB + KBS - 1) / KBS;

  // buffer resources: rows past the live range read as zero; a copy at or past k gets KG_OOB
  const __amdgpu_buffer_rsrc_t ra = kg_rsrc(p.a + (size_t)m0 * p.lda, (long long)(m_end - m0) * p.lda);
  const __amdgpu_buffer_rsrc_t rw = kg_rsrc(p.w + (size_t)n0 * p.k, (long long)(p.n - n0) * p.k);
  const __amdgpu_buffer_rsrc_t rsa = kg_rsrc(p.sfa, (long long)kw * p.sfa_rows * 4);
  const __amdgpu_buffer_rsrc_t rsb = kg_rsrc(p.sfb, (long long)kw * p.n * 4);
  // copy instruction q of this wave covers block rows 8 (q NW + wave) .. + 7, lane l row + (l >> 3) and the chunk
  // that belongs in slot l & 7 (NW is even, so the chunk depends on the wave's parity only)
  const int chunk = ((lane & 7) ^ (((wave & 1) << 2) | (lane >> 4))) << 4;
  unsigned va[QA], vw[QB];
#pragma unroll
  for (int q = 0; q < QA; ++q) va[q] = (unsigned)(((q * NW + wave) * 8 + (lane >> 3)) * p.lda + chunk);
#pragma unroll
  for (int q = 0; q < QB; ++q) vw[q] = (unsigned)(((q * NW + wave) * 8 + (lane >> 3)) * p.k + chunk);
  // copy instruction c (of NQ) of stage s into its buffer
  auto copy1 = [&](u8* st, int s, int c) __attribute__((always_inline)) {
    const int x = c / (QA + QB), q = c % (QA + QB), ko = (s * KBS + x) * 128;
    u8* const blk = st + x * BLK + wave * 1024;
    if (q < QA) kg_ring_copy(ra, blk + q * NW * 1024, ko < p.k ? va[q] : KG_OOB, ko);
    else kg_ring_copy(rw, blk + BM * 128 + (q - QA) * NW * 1024, ko < p.k ? vw[q - QA] : KG_OOB, ko);
  };

  // fragment and scale word offsets: every fragment row is (lane & 31) plus a multiple of 32
  const int arow = wm * TJ * 32 + (lane & 31), wrow = wn * TI * 32 + (lane & 31);
  unsigned offa[2][2], offw[2][2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      const unsigned sw = (unsigned)(((kh * 4 + (lane >> 5) * 2 + h) ^ (((lane & 31) >> 1) & 7)) << 4);
      offa[kh][h] = (unsigned)arow * 128u + sw;
      offw[kh][h] = (unsigned)(BM + wrow) * 128u + sw;
    }
  u32 wa[DW][TJ], wb[DW][TI];
  auto words = [&](int g, int d) __attribute__((always_inline)) {
    // the group's offset is part of the range-checked VGPR offset: a group past the last reads zeros (unused)
    const unsigned ga = (unsigned)(g * p.sfa_rows) * 4u, gb = (unsigned)(g * p.n) * 4u;
#pragma unroll
    for (int j = 0; j < TJ; ++j)
      wa[d][j] = __builtin_amdgcn_raw_buffer_load_b32(rsa, ga + (unsigned)(m0 + arow + j * 32) * 4u, 0, 0);
#pragma unroll
    for (int i = 0; i < TI; ++i)
      wb[d][i] = __builtin_amdgcn_raw_buffer_load_b32(rsb, gb + (unsigned)(n0 + wrow + i * 32) * 4u, 0, 0);
  };

  v16f acc[TI][TJ];
#pragma unroll
  for (int i = 0; i < TI; ++i)
#pragma unroll
    for (int j = 0; j < TJ; ++j)
#pragma unroll
      for (int x = 0; x < 16; ++x) acc[i][j][x] = 0.0f;
  v8i fa[2][U][TJ], fw[2][U][TI];              // [unit parity][half of the unit][tile]
  // fragment f (of NF) of unit u of a stage buffer, in the order the MFMAs first need them
  auto frag1 = [&](const u8* st, int set, int u, int f) __attribute__((always_inline)) {
    const int x = f / (TI + TJ), y = f % (TI + TJ), h = u * U + x;
    const u8* const b = st + (h >> 1) * BLK;
    if (y == 0 || y > TJ) {
      const int i = y == 0 ? 0 : y - TJ;
      fw[set][x][i] = kg_lds_frag(b + i * 4096, offw[h & 1][0], offw[h & 1][1]);
    } else {
      fa[set][x][y - 1] = kg_lds_frag(b + (y - 1) * 4096, offa[h & 1][0], offa[h & 1][1]);
    }
  };
  // One stage s = the loop's base + PH, for a computing wave or one that only copies.
  auto stage = [&](auto ph, auto comp, int s) __attribute__((always_inline)) {
    constexpr int PH = decltype(ph)::value;
    constexpr bool COMP = decltype(comp)::value;
    u8* const cur = buf(ph);
    u8* const prv = buf(std::integral_constant<int, PH + BODY - 1>{});
    const u8* const nxt = buf(std::integral_constant<int, PH + 1>{});
    if constexpr (KBS == 2 && COMP) {
      // two blocks a stage: the scale bytes of a block at or past K are made the unit exponent (its codes are zeros)
#pragma unroll
      for (int x = 0; x < KBS; ++x) {
        if ((PH * KBS + x) % 4 != 0) continue;
        const int live_b = KB - (s * KBS + x), d = (PH * KBS + x) / 4 % DW;
        const u32 keep = live_b >= 4 ? 0xffffffffu : live_b <= 0 ? 0u : (0xffffffffu >> (32 - 8 * live_b));
        const u32 unit = 0x7f7f7f7fu & ~keep;
#pragma unroll
        for (int j = 0; j < TJ; ++j) wa[d][j] = (wa[d][j] & keep) | unit;
#pragma unroll
        for (int i = 0; i < TI; ++i) wb[d][i] = (wb[d][i] & keep) | unit;
      }
    }
    auto slot = [&](auto tt) __attribute__((always_inline)) {
      constexpr int t = decltype(tt)::value, h = t / (TI * TJ), u = h / U, x = h % U, i = t / TJ % TI, j = t % TJ;
      constexpr int set = (PH * UPS + u) & 1, blk = PH * KBS + (h >> 1), d = (blk >> 2) % DW, by = blk & 3;
      if constexpr (COMP) {
        acc[i][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(fw[set][x][i], fa[set][x][j], acc[i][j], 0, 0, by,
                                                                    (int)wb[d][i], by, (int)wa[d][j]);
        __builtin_amdgcn_sched_barrier(0);
        // the second unit's fragments, from this stage's buffer
        if constexpr (UPS == 2 && t < BAR) {
#pragma unroll
          for (int f = t * FR; f < (t == BAR - 1 ? NF : (t + 1) * FR); ++f)
            if (f < NF) frag1(cur, (PH * UPS + 1) & 1, 1, f);
        }
      }
      // the copies of stage s - 1 + NS that did not fit after the last barrier
      if constexpr (t < BAR) {
#pragma unroll
        for (int c = 0; c < CPS; ++c)
          if (C1 + t * CPS + c < NQ) copy1(prv, s - 1 + NS, C1 + t * CPS + c);
      }
      if constexpr (t == BAR) kg_ring_barrier<(NS - 2) * NQ>();
      if constexpr (COMP && t >= BAR) {
        __builtin_amdgcn_sched_barrier(0);
        // the next stage's first unit
#pragma unroll
        for (int f = (t - BAR) * FR; f < (t == NT - 1 ? NF : (t - BAR + 1) * FR); ++f)
          if (f < NF) frag1(nxt, (PH * UPS + UPS) & 1, 0, f);
      }
      if constexpr (t > BAR) {
#pragma unroll
        for (int c = 0; c < CPS; ++c)
          if ((t - BAR - 1) * CPS + c < C1) copy1(cur, s + NS, (t - BAR - 1) * CPS + c);
      }
      // the word group whose last block was in the stage before goes DW groups ahead
      if constexpr (COMP && t == NT - 1 && (PH * KBS) % 4 == 0) {
        constexpr int dn = (PH * KBS / 4 + DW - 1) % DW;
        words((s * KBS >> 2) - 1 + DW, dn);
      }
      __builtin_amdgcn_sched_barrier(0);
    };
    kg_unroll(slot, std::make_integer_sequence<int, NT>{});
  };

  // prologue: the word groups (group DW - 1 goes out in stage 0), then the stages as the loop leaves them
#pragma unroll
  for (int d = 0; d < DW - 1; ++d) words(d, d);
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
  auto fill = [&](auto ss) __attribute__((always_inline)) {
    constexpr int S = decltype(ss)::value;
#pragma unroll
    for (int c = 0; c < (S == NS - 1 ? C1 : NQ); ++c) copy1(buf(ss), S, c);
    __builtin_amdgcn_sched_barrier(0);
  };
  kg_unroll(fill, std::make_integer_sequence<int, NS>{});
  kg_ring_barrier<(NS - 2) * NQ + C1>();
  __builtin_amdgcn_sched_barrier(0);

#define KG_RSTAGE(PH)                                                   \
  if constexpr ((PH) < BODY) {                                          \
    stage(std::integral_constant<int, (PH)>{}, comp, s + (PH));         \
    if (s + (PH) + 1 >= KS) break;                                      \
  }
  auto run = [&](auto comp) __attribute__((always_inline)) {
    if constexpr (decltype(comp)::value) {
#pragma unroll
      for (int f = 0; f < NF; ++f) frag1(st0, 0, 0, f);
      __builtin_amdgcn_sched_barrier(0);
    }
    for (int s = 0;; s += BODY) {
      KG_RSTAGE(0)
      KG_RSTAGE(1)
      KG_RSTAGE(2)
      KG_RSTAGE(3)
      KG_RSTAGE(4)
      KG_RSTAGE(5)
      KG_RSTAGE(6)
      KG_RSTAGE(7)
      KG_RSTAGE(8)
      KG_RSTAGE(9)
      KG_RSTAGE(10)
      KG_RSTAGE(11)
    }
  };
#undef KG_RSTAGE
  // (the waves that only copy run the same barriers in a loop of their own)
  const bool computes = NW == WM * WN || wave < WM * WN;
  if constexpr (NW == WM * WN) {
    run(std::true_type{});
  } else {
    if (computes) run(std::true_type{});
    else run(std::false_type{});
  }
  // no copy may still be writing LDS when the workgroup retires
  asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)" ::: "memory");
  if (!computes) return;

  // lane (lane & 31, lane >> 5) holds columns 8 rr + 4 (lane >> 5) .. + 3 of row (lane & 31) of each MFMA tile
#pragma unroll
  for (int j = 0; j < TJ; ++j) {
    const int row = m0 + arow + j * 32;
    if (row >= m_end) continue;
    u16* const crow = p.c + (size_t)row * p.ldc;
#pragma unroll
    for (int i = 0; i < TI; ++i)
#pragma unroll
      for (int rr = 0; rr < 4; ++rr) {
        const int gn = n0 + wn * TI * 32 + i * 32 + rr * 8 + (lane >> 5) * 4;
        const v16f& v = acc[i][j];
        if (gn + 3 < p.n) {
          uint2 o;
          o.x = kg_pack_bf16x2(v[rr * 4 + 0], v[rr * 4 + 1]);
          o.y = kg_pack_bf16x2(v[rr * 4 + 2], v[rr * 4 + 3]);
          *reinterpret_cast<uint2*>(crow + gn) = o;
        } else {
#pragma unroll
          for (int x = 0; x < 4; ++x)
            if (gn + x < p.n) crow[gn + x] = kg_f32_to_bf16(v[rr * 4 + x]);
        }
      }
  }
}

#define KG_RING_SHAPES(X)                                                                                  \
  X(1, 1, 1, 1, 4, 8, 2, 4, 0, 2, 2)   /* 32 x 32: one wave computes, four copy */                         \
  X(2, 2, 1, 1, 4, 8, 1, 2, 0, 4, 4)   /* 64 x 64 */                                                       \
  X(2, 2, 1, 2, 4, 4, 1, 1, 0, 2, 3)   /* 64 x 128 */                                                      \
  X(4, 2, 1, 2, 8, 4, 1, 1, 0, 2, 2)   /* 128 x 128: eight waves of 32 x 64 (four of 64 x 64 ran 2% slower) */ \
  X(2, 2, 2, 3, 4, 3, 1, 1, 1, 2, 1)   /* 128 x 192 */
#define KG_RING_INSTANCE(...) template __global__ void kg_fp8_gemm_ring<__VA_ARGS__>(const KgFp8Args);
KG_RING_SHAPES(KG_RING_INSTANCE)

template <int... C>
static int kg_ring_go(KgFp8Args& p, hipStream_t st) {
  using R = KgRing<C...>;
  p.m_tiles = (p.m + R::BM - 1) / R::BM, p.n_tiles = (p.n + R::BN - 1) / R::BN;
  hipLaunchKernelGGL((kg_fp8_gemm_ring<C...>), dim3(p.m_tiles * p.n_tiles), dim3(R::THREADS), 0, st, p);
  return (int)hipGetLastError();
}

int kg_fp8_ring_launch(KgFp8Args& p, int bm, int bn, hipStream_t st) {
#define KG_RING_CASE(...) \
  if (bm == KgRing<__VA_ARGS__>::BM && bn == KgRing<__VA_ARGS__>::BN) return kg_ring_go<__VA_ARGS__>(p, st);
  KG_RING_SHAPES(KG_RING_CASE)
  return (int)hipErrorInvalidValue;
}
