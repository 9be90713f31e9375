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
//
// What bounds it at 8192 tokens of the Qwen3-30B-A3B layer: the MFMAs are busy
// for 0.54 of the cycles in gate_up's forward and 0.59 in its input gradient, at
// 1.87 GHz (hardware counters); of the alternating segments the ones that read
// fragments and issue DMAs are the longer, hence the checks kept out of them and
// the offsets formed from one register per operand. The chip's power sets the
// clock: on zero operands the same launches take 390 us instead of 445, and 342
// instead of 430.
#pragma once

#include "gemm_persist.h"

namespace pmoe {

// DMA instructions a wave may have in flight at a wait, two for each unit issued
// after the one that has to have landed.
constexpr int kPpFull = 12;     // six units
constexpr int kPpFullHalf = 8;  // the same, two of the six being A1s not fetched for a next tile that is a half one
constexpr int kPpHalf = 6;      // three units: of a half tile, and of a full one's last phase before a half one

// 256 x 256 tiles of eight 128 x 64 wave tiles; wave row w holds rows 64 w ..
// 64 w + 63 of both 128-row halves.
template <typename Tc_>
struct PpCfg : DmaCfg<256, 256, 128, 64, 2, 64, 1, Tc_> {
  static constexpr int UNIT = 16384;  // bytes of one operand half of a k tile
  static constexpr int ROW_SPAN = 192;
  __device__ static constexpr int wave_row(int wm) { return wm * 64; }
  __device__ static constexpr int row_blk(int i) { return (i >> 1) * 128 + (i & 1) * 32; }
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
  __shared__ __attribute__((aligned(16))) int s_tile[64][4];  // group, m0, m_end, n0 of the block's tiles, a ring
  __shared__ int s_idx[GATH == GA_ROWS ? 2 : 1][GATH == GA_ROWS ? 256 : 1];  // row indices of two tiles

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int wm = wave / Cfg::WAVES_N, wn = wave % Cfg::WAVES_N;
  const bool second = wave >= NW / 2;  // the group that runs half a phase later
  const int groups = p.groups;

  TileWalk<Cfg, GM_ROWS> walk;
  if (!walk.init(p, (EPI == EPI_SWIGLU) ? p.inter : p.N, (EPI == EPI_SWIGLU) ? BN / 2 : BN, s_offs, s_scan, nullptr,
                 nullptr, nullptr, nullptr))
    return;

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
  const uint32_t lda2 = (uint32_t)(p.lda * 2), ldb2 = (uint32_t)(p.ldb * 2);

  // Where the block's tiles lie is worked out for many at once (a lane each, in
  // a ring of 64 entries refilled by halves), and the rows a gathered tile
  // reads are fetched to LDS two tiles ahead: a tile's set-up is then one LDS
  // read and a few multiplications, done in the k loop when the DMAs turn to
  // it. (Searching the group and reading the indices through the scalar cache
  // between the tiles took 2.3 K clocks a tile, 4.9 K with a gather; a tile's k
  // loop takes 30 to 80 K.)
  auto fill_tiles = [&](int first, int n) {
    if (tid < n) {
      const int t = walk.at(first + tid);
      int e[4] = {-1, 0, 0, 0};
      if (t >= 0) {
        const int g = rows_group(s_scan, groups, t / walk.ntiles_n);
        int mt, tn;
        rows_tile(t - s_scan[g] * walk.ntiles_n, s_scan[g + 1] - s_scan[g], walk.ntiles_n, walk.mb, tn, mt);
        e[0] = g;
        e[1] = (g == 0 ? 0 : s_offs[g - 1]) + mt * BM;
        e[2] = s_offs[g];
        e[3] = tn * (EPI == EPI_SWIGLU ? BN / 2 : BN);
      }
#pragma unroll
      for (int x = 0; x < 4; ++x) s_tile[(first + tid) & 63][x] = e[x];
    }
    lds_barrier();
  };
  auto tile_info = [&](int k) {
    TileInfo ti;
    const int* e = s_tile[k & 63];
    ti.group = __builtin_amdgcn_readfirstlane(e[0]);
    ti.m0 = __builtin_amdgcn_readfirstlane(e[1]);
    ti.m_end = __builtin_amdgcn_readfirstlane(e[2]);
    ti.n0 = __builtin_amdgcn_readfirstlane(e[3]);
    ti.k_lo = 0;
    ti.k_hi = p.K;
    return ti;
  };
  // Row indices of tile k (256 of them, 64 per wave; past the table's end: 0)
  auto fetch_rows = [&](int k) {
    if constexpr (GATH == GA_ROWS) {
      if (wave < 4) {
        const int m0 = __builtin_amdgcn_readfirstlane(s_tile[k & 63][1]);
        const BufRsrc rs = make_rsrc(p.a_index + m0, (uint64_t)(p.n_index - m0) * 4);
        dma4(rs, lds_addr(reinterpret_cast<const char*>(&s_idx[k & 1][wave * 64])), (uint32_t)(wave * 64 + lane) * 4);
      }
    }
  };

  // What the DMAs fetch: a tile's place, its descriptors (wave-uniform) and this
  // lane's offsets.
  struct LoadTile {
    TileInfo ti;
    BufRsrc rsA, rsB;
    // Byte offsets of this lane's chunks (kOOB: none). The four of an operand's
    // k tile (two units of two instructions) lie at fixed distances, except
    // for gathered rows and SwiGLU columns (which end inside B, not at its end).
    uint32_t a[GATH == GA_ROWS ? 4 : 1], b[EPI == EPI_SWIGLU ? 2 : 1];
    bool half;  // at most 128 rows: A1 is neither fetched nor read
    // a half tile that is its group's only m-tile: no other tile reads its B, which
    // streams in with non-temporal loads (1200 tokens of the Qwen3-30B-A3B layer:
    // the four GEMMs 592 -> 542 us)
    bool stream;
  };
  auto load_tile = [&](int k, LoadTile& T) {
    const int l = fresh_lane(), kc_row = l >> 3;
    T.ti = tile_info(k);
    const int rows = T.ti.m_end - T.ti.m0;
    T.half = rows <= BM / 2;
    T.stream = T.half && T.ti.m0 == (T.ti.group > 0 ? __builtin_amdgcn_readfirstlane(s_offs[max(T.ti.group, 1) - 1]) : 0);
    const bool any = T.ti.group >= 0;  // past the block's last tile every DMA reads zeros
    const int g = any ? T.ti.group : 0;
    if constexpr (GATH == GA_ROWS) T.rsA = make_rsrc(A0, any ? p.a_bytes : 0);  // the whole gathered storage
    else T.rsA = make_rsrc(A0 + (int64_t)T.ti.m0 * p.lda, (uint64_t)rows * lda2);
    T.rsB = make_rsrc(B0 + (int64_t)g * p.strideB, any ? p.b_bytes : 0);
    // A halves: LDS row r of half h is tile row 128 h + r; rows past the group's
    // end lie past the descriptor's bound
    const int r0 = 8 * wave + kc_row;
    if constexpr (GATH == GA_ROWS) {
#pragma unroll
      for (int x = 0; x < 4; ++x)
        T.a[x] = r0 + 64 * x < rows ? (uint32_t)s_idx[k & 1][r0 + 64 * x] * lda2 + (uint32_t)(kc_k * 2) : kOOB;
    } else {
      T.a[0] = (uint32_t)r0 * lda2 + (uint32_t)(kc_k * 2);
    }
    if constexpr (EPI == EPI_SWIGLU) {
      // N halves: half 0 holds gate columns (LDS row r: tile column r), half 1 the matching up columns
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const int col = T.ti.n0 + r0 + 64 * i;
        T.b[i] = col < p.inter ? (uint32_t)col * ldb2 + (uint32_t)(kc_k * 2) : kOOB;
      }
    } else if constexpr (B_KC) {
      // LDS row r of half n is tile column 64 (r / 32) + 32 n + r % 32 (the end of B is the descriptor's)
      T.b[0] = (uint32_t)(T.ti.n0 + 64 * (r0 >> 5) + (r0 & 31)) * ldb2 + (uint32_t)(kc_k * 2);
    } else {
      // [k][n] unit: 32 k-rows of 256 columns, 2 k-rows per instruction
      const int t_kk = 2 * wave + (l >> 5);
      const int col = T.ti.n0 + 8 * ((l & 31) ^ swz_t(t_kk));
      T.b[0] = col < p.N ? (uint32_t)t_kk * ldb2 + (uint32_t)(col * 2) : kOOB;
    }
  };

  // Unit U of k tile kt of T (0: N0, 1: A0, 2: N1, 3: A1) into the slot of parity par.
  // WHOLE: of a whole k tile, and A1 too (nothing to check).
  auto dma_unit = [&](const LoadTile& T, auto uc, auto whole, int kt, int par) {
    constexpr int U = decltype(uc)::value;
    constexpr bool IS_A = U & 1, WHOLE = decltype(whole)::value;
    constexpr int HALF = U >> 1;
    if (!WHOLE && U == 3 && T.half) return;
    const uint32_t dst = lds0 + (IS_A ? 0 : 4 * UNIT) + (uint32_t)par * (2 * UNIT) + HALF * UNIT + wave * 1024;
    const int k0 = kt * BK;
    uint32_t v[2];
    if constexpr (IS_A || B_KC) {
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        const uint32_t k2 = (uint32_t)(k0 * 2);
        if constexpr (IS_A && GATH == GA_ROWS) v[i] = T.a[2 * HALF + i] + k2;
        else if constexpr (IS_A) v[i] = T.a[0] + (k2 + (uint32_t)(128 * HALF + 64 * i) * lda2);
        else if constexpr (EPI == EPI_SWIGLU) v[i] = T.b[i] + (k2 + (HALF ? (uint32_t)p.inter * ldb2 : 0u));
        else v[i] = T.b[0] + (k2 + (uint32_t)(32 * HALF + 128 * i) * ldb2);
        if constexpr (!WHOLE) v[i] = k0 + BK > p.K && k0 + kc_k >= p.K ? kOOB : v[i];  // the k tail
      }
    } else {
      // k-rows past K lie past the descriptor's bound and read as zero
#pragma unroll
      for (int i = 0; i < 2; ++i) v[i] = __builtin_elementwise_add_sat(T.b[0], (uint32_t)(k0 + 32 * HALF + 16 * i) * ldb2);
    }
    if (!WHOLE && !IS_A && T.stream) dma16x2<NW * 1024, true>(T.rsB, dst, v[0], v[1]);
    else dma16x2<NW * 1024>(IS_A ? T.rsA : T.rsB, dst, v[0], v[1]);
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
  auto mfmas = [&](auto pc) {  // of phase P
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

  const int nk = max((p.K + BK - 1) / BK, 2);  // k tiles of every output tile
  constexpr auto kAny = std::integral_constant<bool, false>();
  constexpr auto kWhole = std::integral_constant<bool, true>();
  LoadTile ld;
  fill_tiles(0, 64);
  fetch_rows(0);
  fetch_rows(1);
  wait_vmcnt<0>();
  lds_barrier();
  load_tile(0, ld);
  TileInfo cur = ld.ti;
  bool half = ld.half;
#pragma unroll
  for (int kt = 0; kt < 2; ++kt)
    static_for<0, 4>([&](auto uc) { dma_unit(ld, uc, kAny, kt, kt); });
  wait_vmcnt<0>();
  lds_barrier();
  read_n(std::integral_constant<int, 0>());
  lds_barrier();  // N0's slot is refilled in phase 0
  int par = 0, tile = 0;
  const int lean_end = (p.K & (BK - 1)) == 0 ? nk - 2 : nk - 3;  // k tiles whose DMAs fetch whole k tiles of this tile

  for (;;) {
#pragma unroll
    for (int i = 0; i < MI; ++i)
#pragma unroll
      for (int j = 0; j < NI; ++j)
#pragma unroll
        for (int r = 0; r < 16; ++r) acc[i][j][r] = 0.0f;
    if (((tile + 2) & 31) == 0) fill_tiles(tile + 2, 32);
    // A tile's indices landed before the previous epilogue in the waves that fetched
    // them, and are read in k tile nk - 2: with two k tiles no phase's barrier lies
    // between.
    if (GATH == GA_ROWS && nk == 2) lds_barrier();
    fetch_rows(tile + 2);
    if (second) swap_groups();
    // Phase P of k tile kt, whose DMAs fetch unit P of k tile lkt (two k tiles
    // on). Ahead of a phase's end lie the units of the next six phases, so a
    // wait for kPpFull leaves the next phase's unit landed (kPpFullHalf: two of
    // the six may be A1s not fetched for a next tile that is a half one).
    //
    // A wait covers the wave's own DMAs; a unit may be read once every wave has
    // waited for its share and a barrier has followed. Every wave waits for all
    // of the next tile's first two k tiles before its epilogue, but between that
    // and the first group's first segment there is no barrier: what that
    // segment reads has to have landed by the last phase's wait. That is A0
    // (N0 is read already), and for a half tile N1 as well, hence kPpHalf in
    // the last phase before one. The later units of those k tiles have the
    // first segment's barrier behind them, so the tile waits for none before
    // phase 6, which gives the epilogue's stores, counted with the loads, six
    // phases.
    // The phases between the first two and the last k tiles (`lean`) check
    // none of that: their reads and DMAs are what a segment's length hangs on
    // (the checks there cost 6 to 10 % of the GEMMs' time).
    auto phase = [&](auto pc, auto lean, int kt, int lkt, bool few) {
      constexpr int P = decltype(pc)::value;
      constexpr bool LEAN = decltype(lean)::value;
      if constexpr (P == 3) {
#pragma unroll
        for (int ks = 0; ks < 4; ++ks) lb[ks] ^= 2 * UNIT;
      }
      if constexpr (P == 0) read_a(std::integral_constant<int, 0>());
      else if constexpr (P == 1) read_n(std::integral_constant<int, 1>());
      else if constexpr (P == 2) read_a(std::integral_constant<int, 1>());
      else read_n(std::integral_constant<int, 0>());
      dma_unit(ld, pc, lean, lkt, par);
      if constexpr (LEAN) {
        wait_vmcnt<kPpFull>();
      } else if (kt > 1 || (P >= 2 && kt == 1)) {
        if (!few) wait_vmcnt<kPpFull>();
        else if (P == 3 && kt == nk - 1) wait_vmcnt<kPpHalf>();
        else wait_vmcnt<kPpFullHalf>();
      }
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));  // lgkmcnt(0)
      swap_groups();
      mfmas(pc);
      swap_groups();
    };
    auto k_tile = [&](auto lean, int kt, int lkt, bool few) {
      static_for<0, 4>([&](auto pc) { phase(pc, lean, kt, lkt, few); });
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) la[ks] ^= 2 * UNIT;
      par ^= 1;
    };
    // A tile of at most 128 rows: two phases a k tile. The first reads A0 and N1,
    // the second the next N0, and they issue the units in the same order
    // (without its own A1s), so that tiles of both kinds follow each other.
    // Three units at least follow the last one each wait is for.
    auto half_k_tile = [&](int kt, int lkt) {
      read_a(std::integral_constant<int, 0>());
      read_n(std::integral_constant<int, 1>());
      dma_unit(ld, std::integral_constant<int, 0>(), kAny, lkt, par);
      if (kt > 0) wait_vmcnt<kPpHalf>();  // the next k tile's N0
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));
      swap_groups();
      mfmas(std::integral_constant<int, 0>());
      swap_groups();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) lb[ks] ^= 2 * UNIT;
      read_n(std::integral_constant<int, 0>());
      static_for<1, 4>([&](auto uc) { dma_unit(ld, uc, kAny, lkt, par); });
      if (kt > 0) wait_vmcnt<kPpHalf>();  // its A0 and N1
      __builtin_amdgcn_s_waitcnt((15) | (7 << 4) | (0 << 8) | (3 << 14));
      swap_groups();
      mfmas(std::integral_constant<int, 1>());
      swap_groups();
#pragma unroll
      for (int ks = 0; ks < 4; ++ks) la[ks] ^= 2 * UNIT;
      par ^= 1;
    };
    // From k tile nk - 2 on the DMAs fetch the next tile's first two.
    if (half) {
#pragma unroll 1
      for (int kt = 0; kt < nk; ++kt) {
        if (kt == nk - 2) load_tile(tile + 1, ld);
        half_k_tile(kt, kt >= nk - 2 ? kt + 2 - nk : kt + 2);
      }
    } else {
#pragma unroll 1
      for (int kt = 0; kt < nk; ++kt) {
        if (kt == 2) {
#pragma unroll 1
          for (; kt < lean_end; ++kt) k_tile(kWhole, kt, kt + 2, false);
        }
        const bool next = kt >= nk - 2;
        if (kt == nk - 2) load_tile(tile + 1, ld);
        k_tile(kAny, kt, next ? kt + 2 - nk : kt + 2, next && ld.half);
      }
    }
    if (!second) swap_groups();  // both groups store together
    wait_vmcnt<0>();             // the next tile's first two k tiles, before the stores join the count
    store_slabs<Cfg, Tout, GM_ROWS, EPI, PACK, SLAB>(acc, stage, cur, p, wm, wn, fresh_lane(), half ? MI / 2 : MI);
    ++tile;
    cur = ld.ti;
    half = ld.half;
    if (cur.group < 0) break;
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
