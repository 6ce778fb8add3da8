// Grouped fp8 GEMMs with the weights in fragment order, for the experts of at most 128 rows (and in small calls for
// every expert, 128 rows at a time; the rule is in kg_fp8_wfrag.hip): the same two grouped
// modes and the same arithmetic as kg_fp8_gemm_wfrag (m-grouped psum; m-grouped gate_up with the fused SiLU-mul-quant
// epilogue), bit for bit.
//
// Why.  Such an expert is bound by the stream of its weights (a byte of them meets at most 128 rows), and what a CU
// streams is what it has in flight.  The persistent kernel keeps 256 accumulators and one workgroup a CU, with 32 to
// 48 KB of weights in flight, and its epilogue has the memory to itself: 5 TB/s.  Here a workgroup owns one
// column tile (256 weight rows) of one expert and half the registers, so that two share a CU: one streams while the
// other starts or ends, and they keep 100 to 200 KB in flight.
//   * A wave owns 64 weight rows (modes 1: 64 columns; 2: 32 gate rows and their 32 up rows) over all the expert's
//     rows.  Weight fragments go from HBM into registers, D stages of 128 K ahead; activations through a ring of NB = 4
//     LDS stages, DA stages ahead (the workgroup's four waves share them).
//   * The weights are loaded non-temporally: each byte is used once (gate_up of 64 tokens 852 us without, 779 with).
//   * Up to 64 rows: 2 MFMA tiles of 32 rows a wave, D = 4, DA = 3.  Up to 128: 4 tiles, D = DA = 2.  Rows past the
//     expert's end are not loaded (zeros).
//   * One barrier a stage: this wave's copies of the next stage have landed (issued DA stages before it; since then that
//     stage's weights and DA - 1 stages' copies and weights, and loads complete in issue order) and its reads of this
//     stage are done.
//   * A stage past K (the scale words hold four) multiplies zeros, as in the persistent kernel, so that even the sign
//     of a zero agrees.
#include "kg_fp8_common.h"
#include "kg_ring.h"

typedef unsigned v4u __attribute__((ext_vector_type(4)));

template <int MODE>
__global__ __launch_bounds__(256, 2) void kg_fp8_gemm_wfew(const KgFp8Args p) {
  static_assert(MODE == 1 || MODE == 2, "grouped modes");
  constexpr int CN = MODE == 2 ? 128 : 256, BUF = 64 * 128;   // output columns a tile; 64 rows of a stage
  __shared__ __attribute__((aligned(1024))) u8 ab0[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab1[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab2[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab3[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab4[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab5[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab6[BUF];
  __shared__ __attribute__((aligned(1024))) u8 ab7[BUF];
  __shared__ float xam[4][128];
  __shared__ u8 xe[128];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int unit = (int)blockIdx.x / p.n_tiles, nt = (int)blockIdx.x - unit * p.n_tiles;
  int g = unit, start, m_end;
  if (p.few == 0) {                                            // unit: the 128 rows from `start`, of the expert there
    start = unit << 7, g = -1;
    for (int e0 = 0; e0 < p.groups && g < 0; e0 += 64) {
      const int e = e0 + lane;
      bool here = false;
      if (e < p.groups) here = (e ? ((p.psum[e - 1] + 127) >> 7) << 7 : 0) <= start && start < p.psum[e];
      const unsigned long long m = __ballot(here);
      if (m) g = e0 + __builtin_ctzll(m);
    }
    if (g < 0) return;                                         // uniform: no expert's rows
    m_end = min(p.psum[g], start + 128);
  } else {                                                     // unit: an expert of at most p.few rows
    start = g ? ((p.psum[g - 1] + 127) >> 7) << 7 : 0, m_end = min(p.psum[g], p.rows);
    if (m_end <= start || p.psum[g] - start > p.few || !kg_wf_split(p, lane)) return;   // uniform: the persistent kernel's
  }
  const int nrows = m_end - start;
  const int half = p.n >> 1, kw = (p.k + 511) >> 9, KB = p.k >> 7, KS = kw << 2, n0 = nt * CN;

  const __amdgpu_buffer_rsrc_t ra = kg_rsrc(p.a + (size_t)start * p.lda, (long long)(nrows - 1) * p.lda + p.k);
  const __amdgpu_buffer_rsrc_t rw = kg_rsrc(p.w + (size_t)g * p.n * p.k, (long long)p.n * p.k);
  const __amdgpu_buffer_rsrc_t rsa = kg_rsrc(p.sfa, (long long)kw * p.sfa_rows * 4);
  const __amdgpu_buffer_rsrc_t rsb = kg_rsrc(p.sfb + (size_t)g * kw * p.n, (long long)kw * p.n * 4);
  // this wave's weight rows: two tiles of 32
  int wr[2];
#pragma unroll
  for (int o = 0; o < 2; ++o) wr[o] = MODE == 2 ? (o ? half : 0) + n0 + wave * 32 : n0 + wave * 64 + o * 32;
  // copy instruction of 8 rows from 8 q: lane l row 8 q + (l >> 3), into slot l & 7 its chunk
  unsigned va[2];
#pragma unroll
  for (int par = 0; par < 2; ++par)
    va[par] = (unsigned)((lane >> 3) * p.lda + (((lane & 7) ^ ((par << 2) | (lane >> 4))) << 4));
  unsigned offa[2][2];
#pragma unroll
  for (int kh = 0; kh < 2; ++kh)
#pragma unroll
    for (int h = 0; h < 2; ++h)
      offa[kh][h] = (unsigned)(lane & 31) * 128u +
                    ((unsigned)((kh * 4 + (lane >> 5) * 2 + h) ^ (((lane & 31) >> 1) & 7)) << 4);

  auto buf = [&](auto i) __attribute__((always_inline)) -> u8* {
    constexpr int x = decltype(i)::value & 7;
    if constexpr (x == 0) return ab0;
    else if constexpr (x == 1) return ab1;
    else if constexpr (x == 2) return ab2;
    else if constexpr (x == 3) return ab3;
    else if constexpr (x == 4) return ab4;
    else if constexpr (x == 5) return ab5;
    else if constexpr (x == 6) return ab6;
    else return ab7;
  };

  auto run = [&](auto nt_c, auto da_c, auto dw_c) __attribute__((always_inline)) {
    constexpr int NT = decltype(nt_c)::value;                             // row tiles of 32
    constexpr int DA = decltype(da_c)::value, D = decltype(dw_c)::value;  // stages ahead: copies, weights
    constexpr int HB = NT / 2, NB = 4, QA = 2 * HB;                  // 64-row buffers a stage; stages; copies
    constexpr int YOUNGER = (DA - 1) * (QA + 8) + 8;
    static_assert(NB > DA && D >= DA && 4 % D == 0 && YOUNGER < 60, "ring");
    v16f acc[2][NT];
#pragma unroll
    for (int o = 0; o < 2; ++o)
#pragma unroll
      for (int j = 0; j < NT; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[o][j][r] = 0.0f;
    v8i wf[D][2][2];                                                      // [stage % D][K half][weight tile]
    u32 wa[2][NT], wb[2][2];

    // copies of stage s (ring slot S): row tiles' 64-row halves of the stage
    auto copy = [&](auto sl, int s) __attribute__((always_inline)) {
      constexpr int S = decltype(sl)::value % NB;
      const int ko = s * 128;
#pragma unroll
      for (int q = 0; q < QA; ++q) {
        const int row = (q >> 1) * 64 + (wave * 2 + (q & 1)) * 8;
        u8* const dst = (q >> 1) ? buf(std::integral_constant<int, S * HB + HB - 1>{})
                                 : buf(std::integral_constant<int, S * HB>{});
        const unsigned v = s < KB ? va[q & 1] + (unsigned)(row * p.lda) : KG_OOB;
        kg_ring_copy(ra, dst + (wave * 2 + (q & 1)) * 1024, v, ko);
      }
    };
    auto wload = [&](int set, int s) __attribute__((always_inline)) {
#pragma unroll
      for (int kh = 0; kh < 2; ++kh)
#pragma unroll
        for (int o = 0; o < 2; ++o) {
          const unsigned v = (s < KB ? (unsigned)(wr[o] * p.k) : KG_OOB) + (unsigned)(lane * 16 + kh * 2048);
          const v4u lo = __builtin_amdgcn_raw_buffer_load_b128(rw, v, (unsigned)s * 4096u, 2 /* nt */);
          const v4u hi = __builtin_amdgcn_raw_buffer_load_b128(rw, v + 1024u, (unsigned)s * 4096u, 2 /* nt */);
          wf[set][kh][o].lo = __builtin_bit_cast(__attribute__((ext_vector_type(4))) int, lo);
          wf[set][kh][o].hi = __builtin_bit_cast(__attribute__((ext_vector_type(4))) int, hi);
        }
    };
    // the scale words of K blocks 4 kg .. + 3 (past K: zeros, made unit exponents before use)
    auto words = [&](int x, int kg) __attribute__((always_inline)) {
#pragma unroll
      for (int j = 0; j < NT; ++j)
        wa[x][j] = __builtin_amdgcn_raw_buffer_load_b32(
            rsa, (unsigned)((start + j * 32 + (lane & 31)) * 4 + kg * p.sfa_rows * 4), 0, 0);
#pragma unroll
      for (int o = 0; o < 2; ++o)
        wb[x][o] = __builtin_amdgcn_raw_buffer_load_b32(rsb, (unsigned)((wr[o] + (lane & 31)) * 4 + kg * p.n * 4), 0, 0);
    };
    auto stage = [&](auto ss, int s) __attribute__((always_inline)) {
      constexpr int S = decltype(ss)::value;                              // s % 4: ring slot, weight set, scale byte
      constexpr int PH = S & 3, G = 0;
      if constexpr (PH == 0) {
        const int live = KB - s;
        const u32 keep = live >= 4 ? 0xffffffffu : live <= 0 ? 0u : 0xffffffffu >> (32 - 8 * live);
        const u32 unit = 0x7f7f7f7fu & ~keep;
#pragma unroll
        for (int j = 0; j < NT; ++j) wa[G][j] = (wa[G][j] & keep) | unit;
#pragma unroll
        for (int o = 0; o < 2; ++o) wb[G][o] = (wb[G][o] & keep) | unit;
      }
      const u8* const lo = buf(std::integral_constant<int, (S % NB) * HB>{});
      const u8* const hi = buf(std::integral_constant<int, (S % NB) * HB + HB - 1>{});
#pragma unroll
      for (int kh = 0; kh < 2; ++kh) {
        __builtin_amdgcn_sched_barrier(0);
        v8i af[NT];
#pragma unroll
        for (int j = 0; j < NT; ++j)
          af[j] = kg_lds_frag((j >> 1 ? hi : lo) + (j & 1) * 4096, offa[kh][0], offa[kh][1]);
#pragma unroll
        for (int j = 0; j < NT; ++j)
#pragma unroll
          for (int o = 0; o < 2; ++o)
            acc[o][j] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(wf[S % D][kh][o], af[j], acc[o][j], 0, 0, PH,
                                                                        (int)wb[G][o], PH, (int)wa[G][j]);
      }
      __builtin_amdgcn_sched_barrier(0);
      if constexpr (PH == 0) words(1, (s >> 2) + 1);
      copy(std::integral_constant<int, (S + DA) % 4>{}, s + DA);
      __builtin_amdgcn_sched_barrier(0);
      wload(S % D, s + D);
      __builtin_amdgcn_sched_barrier(0);
      // the copies of stage s + 1 were issued in stage s + 1 - DA: since then that stage's weights and DA - 1 stages'
      // copies and weights (the scale words only add)
      kg_ring_barrier<YOUNGER>();
      __builtin_amdgcn_sched_barrier(0);
    };
    words(0, 0);
    // as the loop issues them: stage v < 0 the copies of v + DA and the weights of v + D
    auto fill = [&](auto ss) __attribute__((always_inline)) {
      constexpr int V = decltype(ss)::value - D;
      if constexpr (V + DA >= 0) copy(std::integral_constant<int, V + DA>{}, V + DA);
      __builtin_amdgcn_sched_barrier(0);
      wload(V + D, V + D);
      __builtin_amdgcn_sched_barrier(0);
    };
    kg_unroll(fill, std::make_integer_sequence<int, D>{});
    kg_ring_barrier<YOUNGER>();
    __builtin_amdgcn_sched_barrier(0);
    for (int s = 0; s < KS; s += 4) {
      stage(std::integral_constant<int, 0>{}, s);
      stage(std::integral_constant<int, 1>{}, s + 1);
      stage(std::integral_constant<int, 2>{}, s + 2);
      stage(std::integral_constant<int, 3>{}, s + 3);
#pragma unroll
      for (int j = 0; j < NT; ++j) wa[0][j] = wa[1][j];
#pragma unroll
      for (int o = 0; o < 2; ++o) wb[0][o] = wb[1][o];
    }
    // no copy may still be writing LDS when the workgroup retires
    asm volatile("s_waitcnt vmcnt(0) lgkmcnt(0)\n\ts_barrier" ::: "memory");

    if constexpr (MODE == 1) {
      // bf16 through the wave's own 4 KB (its LDS operations execute in order): 16-byte stores, whole 128-byte pieces
      const __amdgpu_buffer_rsrc_t rc = kg_rsrc(p.c, (long long)p.rows * p.ldc * 2);
      u8* const stg = wave < 2 ? ab0 + wave * 4096 : ab1 + (wave - 2) * 4096;
      const int mr = lane & 31;
#pragma unroll
      for (int j = 0; j < NT; ++j) {
#pragma unroll
        for (int o = 0; o < 2; ++o)
#pragma unroll
          for (int rr = 0; rr < 4; ++rr) {
            uint2 v;
            v.x = kg_pack_bf16x2(acc[o][j][rr * 4 + 0], acc[o][j][rr * 4 + 1]);
            v.y = kg_pack_bf16x2(acc[o][j][rr * 4 + 2], acc[o][j][rr * 4 + 3]);
            *reinterpret_cast<uint2*>(stg + mr * 128 + (((o * 4 + rr) ^ (mr & 7)) << 4) + ((lane >> 5) << 3)) = v;
          }
#pragma unroll
        for (int t = 0; t < 4; ++t) {
          const int x = t * 64 + lane, m = x >> 3, c = x & 7, gm = start + j * 32 + m;
          const uint4 v = *reinterpret_cast<const uint4*>(stg + m * 128 + ((c ^ (m & 7)) << 4));
          const unsigned off = gm < m_end ? (unsigned)(gm * p.ldc + n0 + wave * 64 + c * 8) * 2u : KG_OOB;
          const v4u d4 = {v.x, v.y, v.z, v.w};
          __builtin_amdgcn_raw_buffer_store_b128(d4, rc, off, 0, 2 /* nt */);
        }
      }
    } else {
      // SiLU-mul, the row's amax over the four waves' 32 columns each, codes through LDS (row r at 128 r, 16-byte
      // chunk c in slot c ^ (r & 7)), whole 128-byte stores
      float v[NT][16];
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        float am = 0.0f;
#pragma unroll
        for (int r = 0; r < 16; r += 2) {
          kg_silu_mul_acc_bf16x2(acc[0][j][r], acc[1][j][r], acc[0][j][r + 1], acc[1][j][r + 1], v[j][r], v[j][r + 1]);
          am = fmaxf(fmaxf(am, fabsf(v[j][r])), fabsf(v[j][r + 1]));
        }
        am = fmaxf(am, __shfl_xor(am, 32, 64));
        if (lane < 32) xam[wave][j * 32 + lane] = am;
      }
      __syncthreads();
#pragma unroll
      for (int j = 0; j < NT; ++j) {
        const int r = j * 32 + (lane & 31);
        const u32 e = kg_ue8m0(fmaxf(fmaxf(xam[0][r], xam[1][r]), fmaxf(xam[2][r], xam[3][r])), 1e-10f);
        const float inv = kg_exp2i_inv(e);
#pragma unroll
        for (int rr = 0; rr < 4; ++rr) {
          const int col = wave * 32 + rr * 8 + (lane >> 5) * 4;
          *reinterpret_cast<u32*>((j < 2 ? ab0 : ab1) + (r & 63) * 128 + ((((col >> 4) ^ (r & 7)) << 4) | (col & 15))) =
              kg_e4m3x4(v[j][rr * 4] * inv, v[j][rr * 4 + 1] * inv, v[j][rr * 4 + 2] * inv, v[j][rr * 4 + 3] * inv);
        }
        if (wave == 0 && lane < 32) xe[r] = (u8)e;
      }
      __syncthreads();
      const __amdgpu_buffer_rsrc_t rq = kg_rsrc(p.q, (long long)p.rows * half);
      const __amdgpu_buffer_rsrc_t rs = kg_rsrc(p.qsf, (long long)((half + 511) >> 9) * p.sf_rows * 4);
#pragma unroll
      for (int t = 0; t < NT; ++t) {
        const int x = t * 256 + tid, r = x >> 3, c = x & 7, gm = start + r;
        const uint4 v4 = *reinterpret_cast<const uint4*>((t < 2 ? ab0 : ab1) + (r & 63) * 128 + ((c ^ (r & 7)) << 4));
        const v4u d4 = {v4.x, v4.y, v4.z, v4.w};
        __builtin_amdgcn_raw_buffer_store_b128(d4, rq, gm < m_end ? (unsigned)(gm * half + n0 + c * 16) : KG_OOB, 0, 0);
      }
      if (tid < NT * 32) {
        const int gm = start + tid;
        __builtin_amdgcn_raw_buffer_store_b8(
            xe[tid], rs, gm < m_end ? (unsigned)((((nt >> 2) * p.sf_rows + gm) << 2) + (nt & 3)) : KG_OOB, 0, 0);
      }
    }
  };
  if (nrows <= 64) run(std::integral_constant<int, 2>{}, std::integral_constant<int, 3>{}, std::integral_constant<int, 4>{});
  else run(std::integral_constant<int, 4>{}, std::integral_constant<int, 2>{}, std::integral_constant<int, 2>{});
}
template __global__ void kg_fp8_gemm_wfew<1>(const KgFp8Args);
template __global__ void kg_fp8_gemm_wfew<2>(const KgFp8Args);

int kg_fp8_wfew_launch(const KgFp8Args& p, int mode, hipStream_t st) {
  const dim3 grid((unsigned)((p.few ? p.groups : p.rows >> 7) * p.n_tiles));
  if (mode == 1) hipLaunchKernelGGL((kg_fp8_gemm_wfew<1>), grid, dim3(256), 0, st, p);
  else hipLaunchKernelGGL((kg_fp8_gemm_wfew<2>), grid, dim3(256), 0, st, p);
  return (int)hipGetLastError();
}
