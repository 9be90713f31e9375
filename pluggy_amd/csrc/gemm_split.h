// fp32 expert GEMMs on the bf16 matrix cores.
//
// An fp32 value is the exact sum of three bf16 ones, each the rounding (to
// nearest) of what the ones before it left: mid is at most 2^-8 of hi's leading
// power, lo 2^-17. A product of two bf16 values is exact in fp32. The six
// products hi.hi, hi.mid, mid.hi, hi.lo, lo.hi and mid.mid are accumulated, the
// smallest first; left out are mid.lo + lo.mid + lo.lo, at most 2^-24 of the
// leading powers' product (half of an fp32 rounding), of random sign and 2^-27
// of it typically. (With pieces by truncation, which cost the same, they reach
// 2^-21 and always lie on one side.) bf16 MFMAs run 16 times as fast as fp32
// ones on this chip, so six of them take 3/8 of the time, and they round the
// accumulator six times per 16 k where the fp32 ones (2 k each) round it eight
// times, though toward zero where those round to nearest.
//
// Relative error against fp64 of normally distributed operands, by the length n
// of the reduction (on fp32 MFMAs): n 3 3.3e-8 (3.6e-8), 8 3.1e-8 (5.4e-8), 40
// 8.3e-8 (1.15e-7), 128 1.6e-7 (2.0e-7), 512 3.4e-7 (4.1e-7), 2048 7.0e-7
// (8.1e-7). Of one and two products it is 3.4e-8 (2.5e-8 and 3.0e-8), the
// accumulator's rounding alone: tiles of at most kSplitMin reduction rows (an
// expert's weight gradient from so few tokens) take fp32 MFMAs.
//
// Time of the six together at H 512, I 1024, 2048 tokens 804 -> 522 us, at H
// 1024, I 512 1410 -> 788, 8192 tokens of the first 2425 -> 1479 (131 TFLOP/s of
// fp32 products at best, 790 of bf16 ones: like the large bf16 GEMMs, bound by
// the clock the chip can hold); these before the lane order of SplitT, which
// took another 3 to 4 % off the whole pass.
//
// A tile with an operand that its pieces do not hold computes itself again on
// fp32 MFMAs:
//  * Infinities, NaNs and magnitudes that round to a bf16 infinity (from
//    3.396e38) make a piece infinite or NaN, and every output they enter infinite
//    or NaN with it: the accumulators say so, at the end.
//  * bf16 subnormals, which the MFMAs take as they are, end at 2^-133, so below
//    2^-110 bits may be lost. What the third piece is made from is then an fp32
//    subnormal: one class comparison per value, which takes the place of the
//    comparisons that found infinities among the operands (the fp32 forward and
//    the six GEMMs measured the same within 1 %).
#pragma once

#include "gemm.h"

namespace pmoe {

// 64 x 128 blocks of four 32 x 64 wave tiles, 32-deep stages in one LDS buffer
// of three bf16 planes per operand row (208 bytes a row: 16 consecutive rows
// at one chunk fall in 16 distinct 16-byte bank groups). Three blocks share a
// CU: one splits and stages while the others multiply (per wave and stage
// about 660 clocks of splitting against 768 of MFMAs). 128 x 128 blocks, two a
// CU, split less per product but measured 583 and 898 us against 522 and 788:
// their tiles fit the experts' rows and the CU count worse.
struct SplitCfg {
  static constexpr int BM = 64, BN = 128, WM = 32, WN = 64, BK = 32, NT = 256;
  static constexpr int WAVES_N = 2, MI = WM / 32, NI = 2;
  static constexpr int ROW = 208;                // bytes of a staged row: 3 planes x 32 k x 2 bytes + 16
  static constexpr int EPI_LD = WN + 4;          // fp32 staging row of the epilogue (floats)
  static constexpr int LDF = BK + 4;             // floats per staged row of the fp32 loop
  static constexpr int SMEM_BYTES = (BM + BN) * ROW;
  static_assert(4 * 32 * EPI_LD * 4 <= SMEM_BYTES && (BM + BN) * LDF * 4 <= SMEM_BYTES,
                "the epilogue's slabs and the fp32 loop's stage fit");
};

// Reduction rows up to which a tile is computed on fp32 MFMAs alone.
constexpr int kSplitMin = 3;
constexpr int kSubnormal = 0x90, kNonFinite = 0x207;  // v_cmp_class_f32: +-subnormal; NaNs and +-infinity

// Four consecutive k of one row, split: 8 bytes per plane.
struct Split4 {
  uint32_t w[3][2];
  bool inexact = false;  // a value's last piece may not hold all that is left of it
  __device__ __forceinline__ explicit Split4(const u32x4& v) {
#pragma unroll
    for (int h = 0; h < 2; ++h) {
      float a = __uint_as_float(v[2 * h]), b = __uint_as_float(v[2 * h + 1]);  // what is left of two values
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) {
        if (pl == 2) inexact |= __builtin_amdgcn_classf(a, kSubnormal) | __builtin_amdgcn_classf(b, kSubnormal);
        const uint32_t q = cvt_pk_bf16(a, b);
        w[pl][h] = q;
        a -= __uint_as_float(q << 16);
        b -= __uint_as_float(q & 0xffff0000u);
      }
    }
  }
  __device__ __forceinline__ void put(char* dst) const {  // dst: the row's chunk in plane 0
#pragma unroll
    for (int pl = 0; pl < 3; ++pl) *reinterpret_cast<uint64_t*>(dst + pl * 64) = w[pl][0] | ((uint64_t)w[pl][1] << 32);
  }
};

// Stagers: fp32 operand rows to LDS, as split planes (put) or as they are
// (put_f32). R rows x 32 k, 256 threads.
template <int R>
struct SplitKc {  // k-contiguous: 8 chunks of 4 k per row
  static constexpr int PER_T = R * 8 / 256;
  const float* rowp[PER_T];
  u32x4 reg[PER_T];
  template <class RowFn>
  __device__ __forceinline__ void init(RowFn rowptr, int tid) {
#pragma unroll
    for (int i = 0; i < PER_T; ++i) rowp[i] = rowptr((tid + i * 256) >> 3);
  }
  __device__ __forceinline__ void load(int k0, int k_hi, int tid) {
    const int k = k0 + (tid & 7) * 4;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      u32x4 v = {0u, 0u, 0u, 0u};
      if (rowp[i] != nullptr && k < k_hi) v = *reinterpret_cast<const u32x4*>(rowp[i] + k);
      reg[i] = v;
    }
  }
  __device__ __forceinline__ bool put(char* lds, int tid) const {
    bool inexact = false;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const Split4 sp(reg[i]);
      sp.put(lds + ((tid + i * 256) >> 3) * SplitCfg::ROW + (tid & 7) * 8);
      inexact |= sp.inexact;
    }
    return inexact;
  }
  __device__ __forceinline__ void put_f32(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < PER_T; ++i)
      *reinterpret_cast<u32x4*>(lds + ((tid + i * 256) >> 3) * SplitCfg::LDF + (tid & 7) * 4) = reg[i];
  }
};

template <int R>
struct SplitT {  // [k][r]: 4 k-rows x 4 columns per unit
  static constexpr int UNITS = 8 * R / 4, PER_T = (UNITS + 255) / 256;
  // Unit u's k-block and first column. Four consecutive lanes read 64 consecutive
  // bytes of a k-row, and the 32 lanes of a half wave (four column blocks, 16 banks
  // apart, by eight k-blocks of two banks) write all 64 LDS banks once. The six
  // GEMMs with their moves, H 1024, E 32, I 512, top-4: with eight lanes on the
  // k-blocks of one column block (a load touches a row per lane) 917 us at 2048
  // tokens and 468 at 431, so 882 and 407; with eight lanes along a row (loads as
  // good, LDS writes two to a bank) 913 and 469.
  __device__ __forceinline__ static int k_of(int u) { return (u >> 2) & 7; }
  __device__ __forceinline__ static int col_of(int u) { return ((u >> 5) * 4 + (u & 3)) * 4; }
  const float* base;
  int64_t ld;
  int r0, r_hi;
  const int32_t* kidx;
  u32x4 reg[PER_T][4];
  __device__ __forceinline__ void init(const float* b, int64_t ld_, int r0_, int r_hi_, const int32_t* kidx_) {
    base = b; ld = ld_; r0 = r0_; r_hi = r_hi_; kidx = kidx_;
  }
  __device__ __forceinline__ void load(int k0, int k_hi, int tid) {
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int u = tid + i * 256, r = r0 + col_of(u);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const int k = k0 + k_of(u) * 4 + j;
        u32x4 v = {0u, 0u, 0u, 0u};
        if ((UNITS % 256 == 0 || u < UNITS) && k < k_hi && r < r_hi)  // (r_hi is a multiple of 8: whole chunks)
          v = *reinterpret_cast<const u32x4*>(base + (int64_t)(kidx != nullptr ? kidx[k] : k) * ld + r);
        reg[i][j] = v;
      }
    }
  }
  __device__ __forceinline__ u32x4 row(int i, int c) const {
    return u32x4{reg[i][0][c], reg[i][1][c], reg[i][2][c], reg[i][3][c]};
  }
  __device__ __forceinline__ bool put(char* lds, int tid) const {
    bool inexact = false;
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int u = tid + i * 256;
      if (UNITS % 256 == 0 || u < UNITS) {
#pragma unroll
        for (int c = 0; c < 4; ++c) {
          const Split4 sp(row(i, c));
          sp.put(lds + (col_of(u) + c) * SplitCfg::ROW + k_of(u) * 8);
          inexact |= sp.inexact;
        }
      }
    }
    return inexact;
  }
  __device__ __forceinline__ void put_f32(float* lds, int tid) const {
#pragma unroll
    for (int i = 0; i < PER_T; ++i) {
      const int u = tid + i * 256;
      if (UNITS % 256 == 0 || u < UNITS) {
#pragma unroll
        for (int c = 0; c < 4; ++c)
          *reinterpret_cast<u32x4*>(lds + (col_of(u) + c) * SplitCfg::LDF + k_of(u) * 4) = row(i, c);
      }
    }
  }
};

template <bool A_KC, bool B_KC, int GM, int EPI>
__global__ __launch_bounds__(SplitCfg::NT, 3) void grouped_gemm_split_kernel(GemmParams p) {
  typedef SplitCfg Cfg;
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, MI = Cfg::MI, NI = Cfg::NI, ROW = Cfg::ROW;
  static_assert(GM == GM_ROWS || GM == GM_RED, "the expert GEMMs");
  static_assert(!(GM == GM_RED && (A_KC || B_KC)), "GM_RED expects [k][m] and [k][n] operands");
  static_assert(EPI != EPI_SWIGLU || (B_KC && GM == GM_ROWS), "SwiGLU epilogue is the gate_up forward");

  __shared__ __attribute__((aligned(16))) char smem[Cfg::SMEM_BYTES];
  __shared__ int s_scan[1025];
  __shared__ int s_found;

  const int tid = threadIdx.x, lane = tid & 63, wave = tid >> 6;
  const int wm = wave / Cfg::WAVES_N, wn = wave % Cfg::WAVES_N;

  // ---- tile: n-tiles of one m-tile side by side
  const int ntiles_n = (EPI == EPI_SWIGLU) ? (p.inter + BN / 2 - 1) / (BN / 2) : (p.N + BN - 1) / BN;
  const int tn = blockIdx.x % ntiles_n, slot = blockIdx.x / ntiles_n;
  TileInfo ti;
  const float* A = reinterpret_cast<const float*>(p.A);
  const float* B = reinterpret_cast<const float*>(p.B);
  if constexpr (GM == GM_ROWS) {
    int g, r0, re;
    if (!rows_tile_lookup<BM>(p.offs, p.groups, slot, s_scan, &s_found, g, r0, re)) return;
    ti.group = g; ti.m0 = r0; ti.m_end = re; ti.k_lo = 0; ti.k_hi = p.K;
    B += (int64_t)g * p.strideB;
  } else {
    const int mt = (p.M + BM - 1) / BM, g = slot / mt;
    ti.group = g; ti.m0 = (slot % mt) * BM; ti.m_end = p.M;
    ti.k_lo = g == 0 ? 0 : p.offs[g - 1];
    ti.k_hi = p.offs[g];
  }
  ti.n0 = (EPI == EPI_SWIGLU) ? tn * (BN / 2) : tn * BN;

  typename std::conditional<A_KC, SplitKc<BM>, SplitT<BM>>::type sa;
  typename std::conditional<B_KC, SplitKc<BN>, SplitT<BN>>::type sb;
  if constexpr (A_KC) {
    const int m0 = ti.m0, me = ti.m_end;
    sa.init([&](int r) -> const float* {
      return m0 + r < me ? A + (int64_t)(p.a_index != nullptr ? p.a_index[m0 + r] : m0 + r) * p.lda : nullptr;
    }, tid);
  } else {
    sa.init(A, p.lda, ti.m0, ti.m_end, p.a_index);
  }
  if constexpr (B_KC) {
    const int n0 = ti.n0;
    sb.init([&](int c) -> const float* {
      if constexpr (EPI == EPI_SWIGLU) {
        // each wave's 64 columns are 32 gate rows then the matching up rows
        const int gcol = n0 + (c >> 6) * 32 + (c & 31);
        return gcol < p.inter ? B + (int64_t)((c & 32) ? p.inter + gcol : gcol) * p.ldb : nullptr;
      } else {
        return n0 + c < p.N ? B + (int64_t)(n0 + c) * p.ldb : nullptr;
      }
    }, tid);
  } else {
    sb.init(B, p.ldb, ti.n0, p.N, p.b_index);
  }

  f32x16 acc[MI][NI];
  auto clear = [&]() {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
  };
  clear();
  const int klen = ti.k_hi - ti.k_lo, nk = klen > 0 ? (klen + BK - 1) / BK : 0;
  const int frow = lane & 31, fhalf = lane >> 5;

  char* const ta = smem;
  char* const tb = smem + BM * ROW;
  // Short reductions and operands that the pieces do not hold go to fp32 MFMAs.
  bool again = klen <= kSplitMin;
  const int nsplit = again ? 0 : nk;
  if (nsplit > 0) {
    sa.load(ti.k_lo, ti.k_hi, tid);
    sb.load(ti.k_lo, ti.k_hi, tid);
  }
  for (int kt = 0; kt < nsplit; ++kt) {
    again |= sa.put(ta, tid);
    again |= sb.put(tb, tid);
    __syncthreads();
    if (kt + 1 < nsplit) {  // the next stage's loads run under this one's MFMAs
      sa.load(ti.k_lo + (kt + 1) * BK, ti.k_hi, tid);
      sb.load(ti.k_lo + (kt + 1) * BK, ti.k_hi, tid);
    }
#pragma unroll
    for (int ks = 0; ks < BK / 16; ++ks) {
      bf16x8 af[3][MI], bf[3][NI];
#pragma unroll
      for (int pl = 0; pl < 3; ++pl) {
#pragma unroll
        for (int i = 0; i < MI; ++i)
          af[pl][i] = *reinterpret_cast<const bf16x8*>(ta + (wm * Cfg::WM + i * 32 + frow) * ROW + pl * 64 + ks * 32 +
                                                       fhalf * 16);
#pragma unroll
        for (int j = 0; j < NI; ++j)
          bf[pl][j] = *reinterpret_cast<const bf16x8*>(tb + (wn * Cfg::WN + j * 32 + frow) * ROW + pl * 64 + ks * 32 +
                                                       fhalf * 16);
      }
      constexpr int PA[6] = {0, 2, 1, 0, 1, 0}, PB[6] = {2, 0, 1, 1, 0, 0};  // smallest products first
#pragma unroll
      for (int q = 0; q < 6; ++q)
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j)
            acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(af[PA[q]][i], bf[PB[q]][j], acc[i][j], 0, 0, 0);
    }
    __syncthreads();
  }
#pragma unroll
  for (int i = 0; i < MI; ++i)
#pragma unroll
    for (int j = 0; j < NI; ++j)
#pragma unroll
      for (int r = 0; r < 16; ++r) again |= __builtin_amdgcn_classf(acc[i][j][r], kNonFinite);
  if (__syncthreads_or(again)) {
    clear();
    float* const fa = reinterpret_cast<float*>(smem);
    float* const fb = fa + BM * Cfg::LDF;
#pragma unroll 1
    for (int kt = 0; kt < nk; ++kt) {
      sa.load(ti.k_lo + kt * BK, ti.k_hi, tid);
      sb.load(ti.k_lo + kt * BK, ti.k_hi, tid);
      sa.put_f32(fa, tid);
      sb.put_f32(fb, tid);
      __syncthreads();
#pragma unroll 1
      for (int ks = 0; ks < BK / 2; ++ks) {
        float af[MI], bf[NI];
#pragma unroll
        for (int i = 0; i < MI; ++i) af[i] = fa[(wm * Cfg::WM + i * 32 + frow) * Cfg::LDF + ks * 2 + fhalf];
#pragma unroll
        for (int j = 0; j < NI; ++j) bf[j] = fb[(wn * Cfg::WN + j * 32 + frow) * Cfg::LDF + ks * 2 + fhalf];
#pragma unroll
        for (int i = 0; i < MI; ++i)
#pragma unroll
          for (int j = 0; j < NI; ++j) acc[i][j] = __builtin_amdgcn_mfma_f32_32x32x2f32(af[i], bf[j], acc[i][j], 0, 0, 0);
      }
      __syncthreads();
    }
  }
  store_tile<Cfg, float, GM, EPI>(acc, reinterpret_cast<float*>(smem), ti, p, wave, wm, wn, lane);
}

template <bool A_KC, bool B_KC, int GM, int EPI>
hipError_t launch_gemm_split(const GemmParams& p, hipStream_t s) {
  typedef SplitCfg Cfg;
  const int64_t ntn = (EPI == EPI_SWIGLU) ? (p.inter + Cfg::BN / 2 - 1) / (Cfg::BN / 2) : (p.N + Cfg::BN - 1) / Cfg::BN;
  const int64_t slots = GM == GM_ROWS ? (int64_t)(p.M + Cfg::BM - 1) / Cfg::BM + p.groups
                                      : (int64_t)p.groups * ((p.M + Cfg::BM - 1) / Cfg::BM);
  const int64_t grid = slots * ntn;
  if (grid <= 0) return hipSuccess;
  if (grid > 0x7fffffffLL) return hipErrorInvalidValue;
  hipLaunchKernelGGL((grouped_gemm_split_kernel<A_KC, B_KC, GM, EPI>), dim3((unsigned)grid), dim3(Cfg::NT), 0, s, p);
  return hipGetLastError();
}

// The six expert GEMMs on fp32 operands.
inline hipError_t expert_gemm_split(int kind, const GemmParams& p, hipStream_t s) {
  switch (kind) {
    case EG_GATE_UP_FWD: return launch_gemm_split<true, true, GM_ROWS, EPI_SWIGLU>(p, s);
    case EG_DOWN_FWD: return launch_gemm_split<true, true, GM_ROWS, EPI_STORE>(p, s);
    case EG_DOWN_DGRAD: return launch_gemm_split<true, false, GM_ROWS, EPI_SWIGLU_BWD>(p, s);
    case EG_DOWN_WGRAD: return launch_gemm_split<false, false, GM_RED, EPI_STORE>(p, s);
    case EG_GATE_UP_DGRAD: return launch_gemm_split<true, false, GM_ROWS, EPI_STORE>(p, s);
    case EG_GATE_UP_WGRAD: return launch_gemm_split<false, false, GM_RED, EPI_STORE>(p, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pmoe
