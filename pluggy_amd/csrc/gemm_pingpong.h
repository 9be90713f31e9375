// Ping-pong main loop for the 256 x 256 tiles of the expert GEMMs.
//
// Same persistent tile walk, operands and epilogues as gemm_persist.h, with a
// k loop built around two facts measured on MI355X: a CU's LDS DMA moves
// about twice the bytes per second when a lane group reads 128-byte row
// pieces rather than 64-byte ones (so stages are 64 deep), and two waves that
// share a SIMD and both interleave LDS reads with MFMAs leave the matrix pipe
// idle around every block barrier.
//
//  * The eight waves form two groups of four (one wave of each per SIMD), half
//    a phase apart: while one group issues a phase's MFMAs the other reads
//    its next fragments from LDS and issues DMAs, and a barrier swaps them.
//  * A 64-deep k tile is four phases. Its operands are four 16 KiB units: A0,
//    A1 (tile rows 0-127 and 128-255) and N0, N1 (B's halves: the first and
//    second 32 columns of every wave for a k-contiguous B, the first and
//    second 32 k-rows for a [k][n] B). Phase 0 reads A0 and multiplies it with
//    N0 (read one phase ahead), phase 1 reads N1, phase 2 reads A1 (times N0),
//    phase 3 reads the next k tile's N0 (A1 times N1): 8 MFMAs of 32 x 32 x 16
//    per wave and phase, 64 fragment registers.
//  * The ring holds two k tiles (128 KiB). A unit's slot is free one phase
//    after it was read, not when its whole k tile is done: phase 0 refills N0,
//    1 A0, 2 N1, 3 A1, all for two k tiles ahead, so a unit is fetched seven
//    phases before it is read and 96-112 KiB are in flight, as in a ring of
//    four 32-deep stages, but in 128-byte pieces.
#pragma once

#include "gemm_persist.h"

namespace pmoe {

// 256 x 256 tiles of eight 128 x 64 wave tiles; wave row w holds rows 64 w ..
// 64 w + 63 of both 128-row halves.
template <typename Tc_>
struct PpCfg : DmaCfg<256, 256, 128, 64, 2, 64, 1, Tc_> {
  static constexpr int UNIT = 16384;  // bytes of one operand half of a k tile
  static constexpr int ROW_SPAN = 192;
  __device__ static constexpr int wave_row(int wm) { return wm * 64; }
  __device__ static constexpr int row_blk(int i) { return (i >> 1) * 128 + (i & 1) * 32; }
};

// One DMA'd 16 KiB unit: two 1 KiB instructions per wave. off: this lane's
// byte offset at the unit's first k, or kOOB.
struct PpUnit {
  uint32_t off[2];
};

template <class Cfg, typename Tout, bool B_KC, int EPI, int GATH>
__global__ __launch_bounds__(Cfg::NT, 1) void grouped_gemm_pp_kernel(GemmParams p) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, BK = Cfg::BK, NW = Cfg::NW, UNIT = Cfg::UNIT;
  constexpr int MI = Cfg::MI, NI = Cfg::NI;
  static_assert(BM == 256 && BN == 256 && BK == 64 && NW == 8 && MI == 4 && NI == 2, "ping-pong tile shape");
  constexpr bool PACK = sizeof(Tout) == 2 && (EPI == EPI_SWIGLU || EPI == EPI_STORE);
  static_assert(PACK || EPI != EPI_SWIGLU, "the SwiGLU forward stages packed bf16");
  static_assert(sizeof(Tout) == 4 || std::is_same<Tout, typename Cfg::Tc>::value || EPI == EPI_STORE,
                "16-bit outputs of the fused epilogues are in the operands' format");
  static_assert(EPI != EPI_SWIGLU || B_KC, "SwiGLU epilogue layout");
  static_assert(GATH == G_NONE || GATH == GA_ROWS, "gathers: A's rows");

  // [A: parity 0 (A0, A1), parity 1][N: parity 0 (N0, N1), parity 1]
  __shared__ __attribute__((aligned(1024))) char smem[8 * UNIT];
  constexpr int SLAB = PACK ? 16 : 8;
  __shared__ __attribute__((aligned(16))) float s_epi[EpiStage<Cfg, PACK, SLAB>::WORDS];
  __shared__ int s_scan[1025];
  __shared__ int s_offs[1024];

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WAVES_N, wn = wave % Cfg::WAVES_N;
  const bool second = wave >= NW / 2;  // the group that runs half a phase later
  const int groups = p.groups;

  TileWalk<Cfg, GM_ROWS> walk;
  if (!walk.init(p, (EPI == EPI_SWIGLU) ? p.inter : p.N, (EPI == EPI_SWIGLU) ? BN / 2 : BN, s_offs, s_scan, nullptr,
                 nullptr, nullptr, nullptr))
    return;
  const int ntiles_n = walk.ntiles_n, mb = walk.mb;

  const uint32_t lds0 = lds_addr(smem);
  float* stage = s_epi + wave * SLAB * EpiStage<Cfg, PACK, SLAB>::ROW;
  const bf16_t* A0 = reinterpret_cast<const bf16_t*>(p.A);
  const bf16_t* B0 = reinterpret_cast<const bf16_t*>(p.B);

  // k-contiguous units: LDS rows of 64 k (128 bytes), 8 rows per instruction;
  // this lane's chunk of its row, the same in both instructions
  const int kc_k = 8 * ((lane & 7) ^ swz_kc<64>(8 * wave + (lane >> 3)));
  // A lane id the compiler cannot trace: what a tile's set-up and epilogue derive
  // from it is computed there instead of held in registers (and spilled) across
  // the tiles.
  auto fresh_lane = [&]() {
    int l = lane;
    asm volatile("" : "+v"(l));
    return l;
  };
  const uint32_t ldb2 = (uint32_t)(p.ldb * 2);

  // A tile: its place and descriptors (wave-uniform), and this lane's DMA offsets.
  struct LoadTile {
    TileInfo ti;
    BufRsrc rsA, rsB;
  };
  struct Offsets {
    PpUnit a[2];
    PpUnit b[B_KC ? 2 : 1];  // [k][n]: both halves share their offsets (32 k-rows apart)
  };
  constexpr int NOFF = sizeof(Offsets) / 4;
  auto setup = [&](int t, LoadTile& T, Offsets& O) {
    const int l = fresh_lane();
    const int kc_row = l >> 3;
    T.ti.group = 0; T.ti.m0 = 0; T.ti.m_end = 0; T.ti.n0 = 0; T.ti.k_lo = 0; T.ti.k_hi = 0;
    const bf16_t* a_base = A0;
    const bf16_t* b_base = B0;
    uint64_t a_bytes = 0, b_bytes = 0;
    if (t >= 0) {
      const int g = rows_group(s_scan, groups, t / ntiles_n);
      const int lo = g == 0 ? 0 : s_offs[g - 1];
      int tn, mt;
      rows_tile(t - s_scan[g] * ntiles_n, s_scan[g + 1] - s_scan[g], ntiles_n, mb, tn, mt);
      T.ti.group = g; T.ti.m0 = lo + mt * BM; T.ti.m_end = s_offs[g];
      T.ti.n0 = (EPI == EPI_SWIGLU) ? tn * (BN / 2) : tn * BN;
      T.ti.k_hi = p.K;
      b_base = B0 + (int64_t)g * p.strideB;
      b_bytes = p.b_bytes;
      if constexpr (GATH == GA_ROWS) {
        a_bytes = p.a_bytes;  // the whole gathered storage
      } else {
        a_base = A0 + (int64_t)T.ti.m0 * p.lda;
        a_bytes = (uint64_t)(T.ti.m_end - T.ti.m0) * p.lda * 2;
      }
    }
    T.rsA = make_rsrc(a_base, a_bytes);
    T.rsB = make_rsrc(b_base, b_bytes);
    const int rows = T.ti.m_end - T.ti.m0;
    // A halves: LDS row r of half h is tile row 128 h + r
#pragma unroll
    for (int h = 0; h < 2; ++h)
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int rb = 128 * h + 8 * (wave + i * NW);
        const int r = rb + kc_row;
        int64_t src = r;
        if constexpr (GATH == GA_ROWS) {
          // 8 consecutive rows per instruction: their indices come through the
          // scalar cache (uniform addresses, clamped into the table)
          typedef const __attribute__((address_space(4))) int32_t cint;
          cint* ci = (cint*)p.a_index;
          const int64_t last = p.n_index - 1;
          const int m0 = __builtin_amdgcn_readfirstlane(T.ti.m0);
          int tok = 0;
#pragma unroll
          for (int j = 0; j < 8; ++j) {
            const int v = ci[min<int64_t>((int64_t)m0 + rb + j, last)];
            tok = kc_row == j ? v : tok;
          }
          src = tok;
        }
        O.a[h].off[i] = r < rows ? (uint32_t)((src * p.lda + kc_k) * 2) : kOOB;
      }
    if constexpr (B_KC) {
      // N halves: LDS row r of half n is tile column 64 (r / 32) + 32 n + r % 32;
      // with SwiGLU half 0 holds gate columns and half 1 the matching up columns
#pragma unroll
      for (int n = 0; n < 2; ++n)
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int r = 8 * (wave + i * NW) + kc_row;
          int col;
          bool ok;
          if constexpr (EPI == EPI_SWIGLU) {
            col = T.ti.n0 + r;  // 32 columns per wave
            ok = col < p.inter;
            col += n * p.inter;
          } else {
            col = T.ti.n0 + 64 * (r >> 5) + 32 * n + (r & 31);
            ok = col < p.N;
          }
          O.b[n].off[i] = ok ? (uint32_t)(((int64_t)col * p.ldb + kc_k) * 2) : kOOB;
        }
    } else {
      // [k][n] unit: 32 k-rows of 256 columns, 2 k-rows per instruction
      const int t_kk = 2 * wave + (l >> 5);
      const int col = T.ti.n0 + 8 * ((l & 31) ^ swz_t(t_kk));
#pragma unroll
      for (int i = 0; i < 2; ++i)
        O.b[0].off[i] = col < p.N ? (uint32_t)(t_kk + 2 * i * NW) * ldb2 + (uint32_t)(col * 2) : kOOB;
    }
  };

  // Unit U of k tile kt of T (0: N0, 1: A0, 2: N1, 3: A1) into the slot of parity par.
  auto dma_unit = [&](const LoadTile& T, const Offsets& O, auto uc, int kt, int par) {
    constexpr int U = decltype(uc)::value;
    constexpr bool IS_A = U & 1;
    constexpr int HALF = U >> 1;
    const uint32_t dst = lds0 + (IS_A ? 0 : 4 * UNIT) + (uint32_t)par * (2 * UNIT) + HALF * UNIT + wave * 1024;
    const int k0 = kt * BK;
    if constexpr (IS_A || B_KC) {
      const PpUnit& u = IS_A ? O.a[HALF] : O.b[B_KC ? HALF : 0];
      uint32_t v[2] = {u.off[0] + (uint32_t)(k0 * 2), u.off[1] + (uint32_t)(k0 * 2)};
      const bool out = k0 + BK > p.K && k0 + kc_k >= p.K;  // the k tail
      v[0] = out ? kOOB : v[0];
      v[1] = out ? kOOB : v[1];
#pragma unroll
      for (int i = 0; i < 2; ++i) dma16(IS_A ? T.rsA : T.rsB, dst + i * NW * 1024, v[i]);
    } else {
      // k-rows past K lie past the descriptor's bound and read as zero
      const uint32_t base = (uint32_t)(k0 + 32 * HALF) * ldb2;
#pragma unroll
      for (int i = 0; i < 2; ++i) dma16(T.rsB, dst + i * NW * 1024, __builtin_elementwise_add_sat(O.b[0].off[i], base));
    }
  };

  // Lane addresses of the fragments within the operand's LDS region (parity
  // in bit 15, flipped as the k tiles go by). k-contiguous rows: one per
  // substep (the chunk is XORed with the row's swizzle); [k][n]: one per
  // 32-column block.
  uint32_t la[4], lb[4] = {0u, 0u, 0u, 0u};
  {
    const int r = lane & 31, hi = lane >> 5, sw = swz_kc<64>(r);
#pragma unroll
    for (int ks = 0; ks < 4; ++ks) {
      la[ks] = (uint32_t)((wm * 64 + r) * 128 + (((2 * ks + hi) ^ sw) << 4));
      if constexpr (B_KC) lb[ks] = 4 * UNIT + (uint32_t)((wn * 32 + r) * 128 + (((2 * ks + hi) ^ sw) << 4));
    }
    if constexpr (!B_KC) {
#pragma unroll
      for (int j = 0; j < 2; ++j) lb[j] = 4 * UNIT + t_lane_off<256>(wn * 64 + j * 32, lane);
    }
  }
  bf16x8 af[2][4], bfr[2][4];  // A: [32-row block][substep]; B: [32-column block][substep]
  auto read_a = [&](auto hc) {
    constexpr int h = decltype(hc)::value;
#pragma unroll
    for (int ks = 0; ks < 4; ++ks)
#pragma unroll
      for (int i = 0; i < 2; ++i)
        af[i][ks] = *reinterpret_cast<const bf16x8*>(smem + la[ks] + h * UNIT + i * 4096);
  };
  auto read_n = [&](auto nc) {
    constexpr int n = decltype(nc)::value;
    if constexpr (B_KC) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) bfr[n][ks] = *reinterpret_cast<const bf16x8*>(smem + lb[ks] + n * UNIT);
    } else {
#pragma unroll
      for (int ks = 2 * n; ks < 2 * n + 2; ++ks)
#pragma unroll
        for (int j = 0; j < 2; ++j) bfr[j][ks] = t_frag_at<256>(smem, lb[j], ks);
    }
  };

  f32x16 acc[MI][NI];
  auto mfmas = [&](auto pc) {
    constexpr int P = decltype(pc)::value, h = P >> 1, n = P & 1;
    __builtin_amdgcn_s_setprio(1);
    if constexpr (B_KC) {
#pragma unroll
      for (int ks = 0; ks < 4; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
          acc[2 * h + i][n] = mfma16<typename Cfg::Tc>(af[i][ks], bfr[n][ks], acc[2 * h + i][n]);
    } else {
#pragma unroll
      for (int ks = 2 * n; ks < 2 * n + 2; ++ks)
#pragma unroll
        for (int i = 0; i < 2; ++i)
#pragma unroll
          for (int j = 0; j < 2; ++j)
            acc[2 * h + i][j] = mfma16<typename Cfg::Tc>(af[i][ks], bfr[j][ks], acc[2 * h + i][j]);
    }
    __builtin_amdgcn_s_setprio(0);
  };
  // Barrier between segments: the MFMAs and reads of one segment stay on their side of it.
  auto swap_groups = [&]() {
    __builtin_amdgcn_sched_barrier(0);
    asm volatile("" ::: "memory");
    __builtin_amdgcn_s_barrier();
    asm volatile("" ::: "memory");
    __builtin_amdgcn_sched_barrier(0);
  };

  // The next tile's offsets wait in the wave's part of the epilogue's LDS, free
  // while k tiles run: only one set is held in registers.
  static_assert(NOFF * 64 <= SLAB * EpiStage<Cfg, PACK, SLAB>::ROW, "a tile's offsets fit the wave's staging");
  uint32_t* st_off = reinterpret_cast<uint32_t*>(stage) + lane;
  LoadTile cur, nxt, ld;
  Offsets off;
  auto park = [&](const Offsets& O) {
    const uint32_t* o = &O.a[0].off[0];
#pragma unroll
    for (int x = 0; x < NOFF; ++x) st_off[x * 64] = o[x];
  };
  const int nk = max((p.K + BK - 1) / BK, 2);  // k tiles of every output tile
  int tile = 0;
  {
    Offsets o;
    setup(walk.at(1), nxt, o);
    park(o);
  }
  setup(walk.at(0), cur, off);
  ld = cur;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
    static_for<0, 4>([&](auto uc) { dma_unit(ld, off, uc, kt, kt); });
  wait_vmcnt<0>();
  lds_barrier();
  read_n(std::integral_constant<int, 0>());
  lds_barrier();  // N0's slot is refilled in phase 0
  int par = 0;

  for (;;) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    // A row-grouped tile of at most 128 rows needs A0 alone: two phases a k tile.
    const bool half = cur.ti.m_end - cur.ti.m0 <= BM / 2;
    if (second) swap_groups();
    // Phase P of k tile kt, whose DMAs fetch unit P of k tile lkt of T (two k
    // tiles on). Ahead of a phase's end lie the units of the next six phases,
    // two instructions each, so a wait for vmcnt(12) leaves the next phase's
    // unit landed. A tile's first seven units landed before its first phase
    // (the prologue, or the wait before the epilogue): no wait until phase 6,
    // which gives the epilogue's stores, counted with the loads, six phases.
    auto phase = [&](auto pc, int kt, int lkt) {
      constexpr int P = decltype(pc)::value;
      if constexpr (P == 3) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) lb[ks] ^= 2 * UNIT;
      }
      if constexpr (P == 0) read_a(std::integral_constant<int, 0>());
      else if constexpr (P == 1) read_n(std::integral_constant<int, 1>());
      else if constexpr (P == 2) read_a(std::integral_constant<int, 1>());
      else read_n(std::integral_constant<int, 0>());
      dma_unit(ld, off, pc, lkt, par);
      if (kt > 1 || (P >= 2 && kt == 1)) wait_vmcnt<12>();
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
      swap_groups();
      mfmas(pc);
      swap_groups();
    };
    auto k_tile = [&](int kt, int lkt) {
      static_for<0, 4>([&](auto pc) { phase(pc, kt, lkt); });
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) la[ks] ^= 2 * UNIT;
      par ^= 1;
    };
    // The half tile's k tile: its two phases read A0 and N1, then the next N0,
    // and issue the four units in the same order (A1's rows read zero), so that
    // tiles of both kinds follow each other.
    auto half_k_tile = [&](int kt, int lkt) {
      read_a(std::integral_constant<int, 0>());
      read_n(std::integral_constant<int, 1>());
      dma_unit(ld, off, std::integral_constant<int, 0>(), lkt, par);
      if (kt > 0) wait_vmcnt<8>();  // the next k tile's N0
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));
      swap_groups();
      mfmas(std::integral_constant<int, 0>());
      swap_groups();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) lb[ks] ^= 2 * UNIT;
      read_n(std::integral_constant<int, 0>());
      static_for<1, 4>([&](auto uc) { dma_unit(ld, off, uc, lkt, par); });
      if (kt > 0) wait_vmcnt<10>();  // its A0 and N1
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));
      swap_groups();
      mfmas(std::integral_constant<int, 1>());
      swap_groups();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) la[ks] ^= 2 * UNIT;
      par ^= 1;
    };
    // From k tile nk - 2 on the DMAs fetch the next tile's first two.
    auto to_next = [&]() {
      ld = nxt;
      uint32_t* o = &off.a[0].off[0];
#pragma unroll
      for (int x = 0; x < NOFF; ++x) o[x] = st_off[x * 64];
    };
    if (half) {
#pragma unroll 1
      for (int kt = 0; kt < nk; ++kt) {
        if (kt == nk - 2) to_next();
        half_k_tile(kt, kt < nk - 2 ? kt + 2 : kt + 2 - nk);
      }
    } else {
#pragma unroll 1
      for (int kt = 0; kt < nk; ++kt) {
        if (kt == nk - 2) to_next();
        k_tile(kt, kt < nk - 2 ? kt + 2 : kt + 2 - nk);
      }
    }
    if (!second) swap_groups();  // both groups store together
    wait_vmcnt<0>();             // the next tile's first two k tiles, before the stores join the count
    store_slabs<Cfg, Tout, GM_ROWS, EPI, PACK, SLAB>(acc, stage, cur.ti, p, wm, wn, fresh_lane(), half ? MI / 2 : MI);
    ++tile;
    if (walk.at(tile) < 0) break;
    cur = nxt;
    Offsets o;
    setup(walk.at(tile + 1), nxt, o);
    park(o);  // (after the epilogue's reads, in the wave's LDS order)
  }
  wait_vmcnt<0>();  // the zero-reading DMAs past the last tile
}

template <class Cfg, bool B_KC, int EPI, int GATH = G_NONE, typename Tout = typename Cfg::Tc>
hipError_t launch_gemm_pp(const GemmParams& p, int num_cus, hipStream_t s) {
  if (p.groups > 1024) return hipErrorInvalidValue;
  const int grid = num_cus > 0 ? num_cus : 256;
  hipLaunchKernelGGL((grouped_gemm_pp_kernel<Cfg, Tout, B_KC, EPI, GATH>), dim3(grid), dim3(Cfg::NT), 0, s, p);
  return hipGetLastError();
}

// The row-grouped expert GEMMs (forward and dgrad) on the ping-pong kernel.
template <class Cfg, typename T16 = typename Cfg::Tc>
hipError_t expert_gemm_pp_rows(int kind, const T16* A, const T16* B, const T16* aux, T16* C, T16* C2,
                               const int32_t* offs, int P, int E, int H, int I, const ExpertGather& xg, int num_cus,
                               hipStream_t s) {
  const GemmParams p = expert_params(kind, A, B, aux, C, C2, offs, P, E, H, I, xg);
  const bool gath = xg.index != nullptr;
  switch (kind) {
    case EG_GATE_UP_FWD:
      if (gath) return launch_gemm_pp<Cfg, true, EPI_SWIGLU, GA_ROWS>(p, num_cus, s);
      return launch_gemm_pp<Cfg, true, EPI_SWIGLU>(p, num_cus, s);
    case EG_DOWN_FWD: return launch_gemm_pp<Cfg, true, EPI_STORE>(p, num_cus, s);
    case EG_DOWN_DGRAD:
      if (gath) return launch_gemm_pp<Cfg, false, EPI_SWIGLU_BWD, GA_ROWS>(p, num_cus, s);
      return launch_gemm_pp<Cfg, false, EPI_SWIGLU_BWD>(p, num_cus, s);
    case EG_GATE_UP_DGRAD: return launch_gemm_pp<Cfg, false, EPI_STORE>(p, num_cus, s);
  }
  return hipErrorInvalidValue;
}

}  // namespace pmoe
