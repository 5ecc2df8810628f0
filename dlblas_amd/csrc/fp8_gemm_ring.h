// Compute-bound FP8 block-scaled GEMM for gfx950: tiles streamed HBM -> LDS by the DMA path into a ring of K steps, eight
// waves (two per SIMD), 16 x 16 x 128 e4m3 MFMA, block scales applied with one FMA per accumulator element and K step.
//
// What bounds it: the power limit.  Over a long K the chip settles at 1.7 to 1.9 of its 2.4 GHz, so a K step costs its energy
// as well as its stalls, and every choice below is about one of the two:
//   - 16 x 16 x 128 instead of two chained 32 x 32 x 64: the same bits (see chunk0), but
//     8 % less time at the power limit (a loop of nothing but MFMAs and scale FMAs on random codes: 3593 against 3322 TFLOP/s,
//     bench.py --ceilings), and a partial sum is 4 registers that are complete two instructions later, instead of 16.  The registers saved hold a
//     ring of streamed fragments, read from LDS three fragments ahead of their use.
//   - two points of a K step at which LDS is handed over instead of one: behind the first, the held operand's rows and the first
//     half of the streamed operand's may be refilled, behind the second the rest.  A byte is on its way for 1.1 K steps or
//     more, where a single hand-over leaves the last of a group 0.4.  Loads are issued one in two MFMA slots; in one burst
//     they cost 3 %.
//   - fragments take every other group of four rows, so that a lane's two results of a pair of fragments are 8 consecutive
//     columns: results go from the registers to memory in 16-byte pieces, 128 or 256 bytes of a row per instruction (lanes exchange chunks
//     through DPP first).  No LDS
//     is involved, so the ring runs on from tile to tile (AHEAD) in every layout but plain contiguous rows.  A tile with the quantising epilogue shares
//     nothing but its rows' largest magnitudes through LDS, where the whole tile used to pass in bf16.
// 4096 x 8192 x 18432 in 256 x 256 tiles: 505 us with 32 x 32 MFMAs and one hand-over per step, 471 us in this form
// (2.62 PFLOP/s); its K steps take 2740 cycles of which 2048 are MFMA.  Without the scale FMAs it would be 421 us.  (All before
// ring_swizzle had its present form, which is worth 2 % more.)
// Expert-contiguous lists, 32 experts, 8192 rows, 4096 x 7168: 330 us per call with the former kernels (32 x 32 MFMAs, results
// through LDS, a ring that drained between tiles), 306 us with these; the whole expert MLP on 8192 tokens 589 -> 532 us, of
// which the ring that runs on is 5.
//
// Arithmetic: fp8_gemm_kernel of the reference (dlblas/kernels/fp8_gemm.py:49-60).  Requires K % 128 == 0.
#pragma once

#include "fp8_gemm_pipelined.h"

namespace dlb {

// WGM x WGN waves, each with MF x NF fragments of 16 x 16 outputs (both even); STAGES K steps of 128 in the ring.
// SCTAB: the activation scales of a tile's rows for all K blocks (at most SCTAB_KB) lie in a table behind the ring, fetched
// once per tile: a row-major a_s then needs no re-layout launch in front.
template <int WGM_, int WGN_, int MF_, int NF_, int STAGES_, bool SCTAB_ = false, int SCTAB_KB_ = 0>
struct RingCfg {
  static constexpr int WGM = WGM_, WGN = WGN_, MF = MF_, NF = NF_, STAGES = STAGES_;
  static constexpr bool SCTAB = SCTAB_;
  static constexpr int WAVES = WGM * WGN, NT = WAVES * 64;
  static constexpr int BM = WGM * MF * 16, BN = WGN * NF * 16;
  static constexpr bool UNIFORM_W = 128 % (NF * 16) == 0;  // a wave's columns share one weight scale
  static constexpr int A_INST = BM / 64, B_INST = BN / 64;  // 16-byte DMA instructions per wave and K step
  static constexpr int L = A_INST + B_INST + 1;             // ... and one for the scales
  static constexpr int A_BYTES = BM * kScaleBlock, B_BYTES = BN * kScaleBlock;
  static constexpr int S_WAVES = SCTAB ? 0 : BM / 64;  // waves whose scale instruction fetches activation scales; the others fetch the weights'
  static constexpr int AS_OFF = A_BYTES + B_BYTES, WS_OFF = AS_OFF + S_WAVES * 256;
  static constexpr int STAGE_BYTES = WS_OFF + 256;
  static constexpr int SCTAB_KB = SCTAB_KB_;
  static constexpr int SCTAB_OFF = STAGES * STAGE_BYTES;
  static constexpr int SCTAB_BYTES = SCTAB ? BM * (SCTAB_KB + 1) * 4 : 0;  // rows of an odd pitch
  static constexpr int ROWS_OFF = SCTAB_OFF + SCTAB_BYTES;  // source rows of the next tile (gathered activations)
  static constexpr int AMAX_OFF = ROWS_OFF + BM * 4;        // largest magnitudes of a tile's rows, per wave column (quantising epilogue)
  static constexpr int LDS_BYTES = SCTAB_OFF + SCTAB_BYTES;
  static constexpr int ACT_LDS_BYTES = AMAX_OFF + BM * WGN * 4;
  // the operand with fewer fragments is held in registers for a K step, the other one streamed past it
  static constexpr bool HOLD_X = MF <= NF;
  static constexpr int H = HOLD_X ? MF : NF, S = HOLD_X ? NF : MF, STRIPS = HOLD_X ? WGN : WGM;
  static constexpr int H_INST = HOLD_X ? A_INST : B_INST, S_INST = HOLD_X ? B_INST : A_INST;
  static constexpr int NB = S % 4 == 0 ? 4 : 3, PD = NB - 1;  // ring of streamed fragments, read PD of them ahead
  // Parts of a K step's DMA group: the held operand, the first LOW streamed fragments of every wave and the scales go into
  // the first part, the rest into the second.
  static constexpr int LOW = S == 6 ? 2 : 4, LOW_INST = STRIPS * LOW * 16 / 64;
  static constexpr int P1 = H_INST + LOW_INST + 1, P2 = L - P1;
  static constexpr int T = H * S;                                  // MFMA slots of a K step
  static constexpr int B1 = H - 1, B2 = H * (S - 1 - PD) + H - 1;  // slots in front of which the parts' LDS is handed over
  static constexpr bool ONE_POINT = B1 == B2;
  static_assert(WAVES == 8 && MF % 2 == 0 && NF % 2 == 0 && (H == 4 || (H == 2 && S == 4)) && (S == 4 || S == 6 || S == 8), "the shapes this is written for");
  static_assert(S % NB == 0 && STRIPS * LOW % 4 == 0 && (ONE_POINT ? P2 == 0 : PD <= LOW), "fragments of a part are there when they are read");
  static_assert(LDS_BYTES <= 160 * 1024, "ring and table fit the LDS");
};

// XOR pattern of the 16-byte chunk index in a 128-byte LDS row.  A ds_read_b128 goes through the 64 banks in four turns of 16 lanes that
// are no neighbours: lanes 0-3, 12-15 and 20-27 take the first, the rest of lanes 0-31 the second.  A fragment's 16 rows are
// four runs of four, eight rows apart, lanes 16-31 read the chunk two further on: with row bit 1 on chunk bit 1 and the run on bits
// 0 and 2, no two lanes of a turn meet in a bank.  With row bit 1 on bit 0 and the run on bits 1 and 2, where 16 neighbouring lanes have no
// conflict, every read took eight turns: SQ_LDS_BANK_CONFLICT 47 % of SQ_LDS_IDX_ACTIVE, now 0; 4096 x 7168 x 18432 441 -> 431 us,
// 4096 x 24576 x 1536 with the quantiser 166 -> 162.
__device__ __forceinline__ int ring_swizzle(int row) { return (row & 2) | ((row >> 3) & 1) | ((row >> 2) & 4); }
// row of a wave's operand that lane or result index i (0 .. 15) of fragment f stands for
__device__ __forceinline__ int ring_row(int f, int i) { return (f >> 1) * 32 + (f & 1) * 4 + (i >> 2) * 8 + (i & 3); }

// Lanes that differ in bit BIT (1 or 2) of their number exchange: a lane with the bit clear gets both lanes' `a`, one with it
// set both lanes' `b`; `a` is then of the lane with the bit clear, `b` of the other.  Every lane has to be active.
template <int BIT>
__device__ __forceinline__ void swap_chunks(v4i& a, v4i& b, int lane) {
  const bool set = lane & BIT;
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const int got = __builtin_amdgcn_update_dpp(0, set ? a[i] : b[i], BIT == 1 ? 0xB1 : 0x4E, 0xF, 0xF, true);  // quad_perm 1,0,3,2 or 2,3,0,1
    a[i] = set ? got : a[i];
    b[i] = set ? b[i] : got;
  }
}

// The same for bit BIT (16 or 32) of the lane number.
template <int BIT>
__device__ __forceinline__ void swap_far_chunks(v4i& a, v4i& b) {
#pragma unroll
  for (int i = 0; i < 4; ++i) {
    const unsigned ua = static_cast<unsigned>(a[i]), ub = static_cast<unsigned>(b[i]);
    if constexpr (BIT == 16) {
      const auto s = __builtin_amdgcn_permlane16_swap(ua, ub, false, false);
      a[i] = static_cast<int>(s[0]), b[i] = static_cast<int>(s[1]);
    } else {
      const auto s = __builtin_amdgcn_permlane32_swap(ua, ub, false, false);
      a[i] = static_cast<int>(s[0]), b[i] = static_cast<int>(s[1]);
    }
  }
}

// Workgroup barrier that orders LDS traffic only (see lds_barrier), as builtins: the compiler then knows that no LDS read is out.
// The waits that it places in a K step are for all reads nevertheless (lgkmcnt(0) ahead of slots 0, 16 and 29 of the 256 x 256 loop, beside
// those of the two barriers): the scale load of a group (dma_4) is the form of load that its model counts on the LDS counter as well,
// and reads behind one are no longer in order for it.  At slot 0 that waits for held fragments of which the last is needed at slot 3.
__device__ __forceinline__ void ring_barrier() {
  __builtin_amdgcn_sched_barrier(0);
  __builtin_amdgcn_s_waitcnt(0xC07F);  // lgkmcnt(0)
  asm volatile("" ::: "memory");
  __builtin_amdgcn_s_barrier();
  asm volatile("" ::: "memory");
  __builtin_amdgcn_sched_barrier(0);
}

// wait_vmcnt<N>() unless `left` (wave-uniform) is above LIMIT.  The branch is hidden in the asm: as control flow inside a K step it would cut the
// step's code into blocks across which nothing is scheduled and registers spill.
template <int N, int LIMIT>
__device__ __forceinline__ void wait_vmcnt_unless(int left) {
  static_assert(N < 64, "vmcnt is a 6-bit counter");
#ifdef __HIP_DEVICE_COMPILE__
  asm volatile("s_cmp_gt_i32 %0, %2\n\ts_cbranch_scc1 1f\n\ts_waitcnt vmcnt(%1)\n1:" ::"s"(__builtin_amdgcn_readfirstlane(left)), "i"(N), "i"(LIMIT) : "memory", "scc");
#endif
}

struct RingTile {
  int g, m0, n0, m_end, split, lin;
};

// Tile lists: the region is entries [lists.first, lists.first + lists.count) of a list's tiles (an entry per row tile and column tile), or, with 64-row tiles,
// the entries' 64-row pieces, lists.pieces each.
struct ListRegion {
  int which, first, count, pieces;
};

// Work of one workgroup: tiles vb_first, vb_first + gridDim.x, ... of a region that is tiles_m x tiles_n tiles of BM x BN and
// starts at column n_base of the output (tile lists: of `lists`).
// AHEAD: the ring runs on from tile to tile; the steps of a tile whose fetches lie past the end of K fetch the first K blocks of
// the workgroup's next tile.
// ODD: bf16 results whose rows lie off dwords (dense, K in one piece).
template <class Cfg, int MODE, bool AHEAD, bool ODD = false>
__device__ __forceinline__ void ring_body(const Args& p, uint8_t* smem, int vb_first, int tiles_m, int tiles_n, int n_base, ListRegion lists = {}) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, MF = Cfg::MF, NF = Cfg::NF, STAGES = Cfg::STAGES, H = Cfg::H, S = Cfg::S, L = Cfg::L;
  constexpr bool kList = MODE == kContigList || MODE == kContigListAct;
  constexpr bool kAct = MODE == kContigListAct || MODE == kMaskedAct;
  constexpr bool kMaskedLike = MODE == kMasked || MODE == kMaskedAct;
  constexpr bool kUniformW = Cfg::UNIFORM_W;
  constexpr int NS = kAct ? 2 : kUniformW ? 1 : NF / 2;  // weight scales of a wave: gate and up, one, or one per 32 columns
  constexpr auto ns_of = [](int ni) { return kAct ? (ni >= NF / 2 ? 1 : 0) : kUniformW ? 0 : ni / 2; };
  // Grouped modes: an expert's weight tile is read by the one to three row tiles of that expert, not by a column of the grid: streamed.
  constexpr int kWeightPolicy = MODE == kDense ? kDmaKeep : kDmaStream;
  static_assert(!kAct || (BN == 256 && kUniformW && !Cfg::SCTAB), "the fused activation pairs 128 gate columns with 128 up columns");

  const int tid = threadIdx.x, lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l16 = lane & 15, q = lane >> 4;
  const lds_bytes_t lds = (lds_bytes_t)smem;  // destination of the DMA: an address in LDS from the start, not a generic one cast at each load
  const int wm0 = (wave / Cfg::WGN) * (MF * 16), wn0 = (wave % Cfg::WGN) * (NF * 16);
  const uint32_t uK = static_cast<uint32_t>(p.K);

  // ---- tiles ------------------------------------------------------------------------------------------------
  const int tiles = tiles_m * tiles_n;
  // Unit id of a dense launch: the tile, in patches of group_m row tiles, and the slice of K; slices of one tile are far apart.
  const int units = MODE == kDense && !AHEAD && !ODD ? tiles * p.splitk : tiles;
  int walk_g = 0, walk_base = 0;
  // tables of a launch's tiles, written by the launch before: scalar loads
  typedef const __attribute__((address_space(4))) int32_t* table_ptr;
  auto entry = [](const int32_t* table, int i) __attribute__((always_inline)) { return reinterpret_cast<table_ptr>(reinterpret_cast<uintptr_t>(table))[i]; };
  // tile number vb of this launch; false: there is none
  auto find = [&](int vb, RingTile& t) __attribute__((always_inline)) {
    int g = 0, mt = 0, nt = 0, m_first = -1;
    t.split = 0, t.lin = 0, t.m_end = p.M;
    if (kMaskedLike) {
      // The tile count is only known on the device, so the grid is persistent; the hardware deals consecutive
      // workgroups to the 8 XCDs in turn.  Of every 32 consecutive tiles each XCD takes 4 consecutive ones: the row
      // tiles of an expert, which are adjacent in the order and read the same weight tile, meet in one L2, and the
      // last, partial round still spreads over all XCDs (the grid is a multiple of 32).
      const int grid = static_cast<int>(gridDim.x);
      const int w = vb % grid;
      const int tile_id = vb - w + (w / 32) * 32 + (w % 8) * 4 + (w / 8) % 4;
      int valid = 0, mtiles = 0;
      while (walk_g < p.G) {
        valid = min(max(entry(p.gidx, walk_g), 0), p.M);
        mtiles = (valid + BM - 1) / BM;
        const int cnt = mtiles * tiles_n;
        if (tile_id < walk_base + cnt) break;
        walk_base += cnt;
        ++walk_g;
      }
      if (walk_g >= p.G) return false;
      g = walk_g;
      const int local = tile_id - walk_base;
      mt = local % mtiles;
      nt = local / mtiles;
      t.m_end = valid;
    } else if (kList) {
      // tiles of this height come from the list the pre-pass built: entry = first 128-row block of the tile.  The
      // column tiles of one row block are adjacent in the order, so they share the activation tile in L2.
      static_assert(!kList || BM == 256 || BM == 192 || BM == 128 || BM == 64, "tile heights of the three lists and their pieces");
      constexpr bool kPieces = BM == 64;
      const int which = kPieces ? lists.which : BM == 256 ? 0 : (BM == 192 ? 1 : 2);
      const int total = kPieces ? lists.count * lists.pieces : lists.count;
      if (vb >= total) return false;
      int v = xcd_remap(vb, total);
      int piece = 0;
      if (kPieces) {
        const int w = v / lists.pieces;  // a tile's pieces side by side: they share its weights in one L2
        piece = v - w * lists.pieces;
        v = w;
      }
      v += lists.first;
      int li;
      if (which == 1) {
        // the two tiles of a pair side by side for every column tile: neighbours in the order run on one XCD at the same time
        const int pair = v / (2 * tiles_n), r = v - pair * 2 * tiles_n;
        nt = r >> 1;
        li = 2 * pair + (r & 1);
      } else {
        li = v / tiles_n;
        nt = v - li * tiles_n;
      }
      m_first = entry(p.tlist, kTileListHeader + which * p.tlist_cap + li) * 64;
      g = entry(p.gidx, m_first);
      m_first = min(m_first + piece * 64, p.M - 1);  // a piece past the end of a short last block: its last row once more
      t.m_end = min(p.M, m_first + BM);
    } else {
      if (vb >= units) return false;
      const int id = xcd_remap(vb, units);
      t.split = MODE == kDense && !AHEAD && !ODD ? id / tiles : 0;
      t.lin = id - t.split * tiles;
      const int width = p.group_m * tiles_n;
      const int grp = t.lin / width;
      const int first_m = grp * p.group_m;
      const int gsz = min(tiles_m - first_m, p.group_m);
      const int in_grp = t.lin - grp * width;
      mt = first_m + in_grp % gsz;
      nt = in_grp / gsz;
      if (MODE == kContiguous) g = entry(p.gidx, mt * BM);
    }
    t.g = __builtin_amdgcn_readfirstlane(g);
    t.m0 = __builtin_amdgcn_readfirstlane(kList ? m_first : mt * BM);
    t.n0 = __builtin_amdgcn_readfirstlane(kAct ? nt * (BN / 2) : n_base + nt * BN);  // kAct: the tile's first OUTPUT column
    return true;
  };

  // ---- DMA addressing ---------------------------------------------------------------------------------------
  // An instruction moves 8 rows; lane i fills chunk (i & 7) of row (i >> 3), which holds the row's chunk (i & 7) ^ pattern.
  // Offsets count from the tile's first row and are held within the rows there are by the descriptor: rows past the end read as
  // zero and cost no traffic.
  // group of 8 rows that instruction j of this wave moves, held operand / streamed operand (first part: the first LOW fragments
  // of every strip); all agree in (group & 3), so the chunk pattern depends on the wave alone
  auto held_row = [&](int j) __attribute__((always_inline)) { return (j * 8 + wave) * 8; };
  auto strm_row = [&](int j) __attribute__((always_inline)) {
    constexpr int kLowG = Cfg::LOW * 2, kUpG = (S - Cfg::LOW) * 2 > 0 ? (S - Cfg::LOW) * 2 : 1;
    const bool low = j < Cfg::LOW_INST;
    const int idx = (low ? j : j - Cfg::LOW_INST) * 8 + wave;
    const int strip = idx / (low ? kLowG : kUpG);
    return strip * S * 16 + (low ? 0 : Cfg::LOW * 16) + (idx - strip * (low ? kLowG : kUpG)) * 8;
  };
  auto a_row = [&](int j) __attribute__((always_inline)) { return Cfg::HOLD_X ? held_row(j) : strm_row(j); };
  auto b_row = [&](int j) __attribute__((always_inline)) { return Cfg::HOLD_X ? strm_row(j) : held_row(j); };
  // kAct: the weight rows of a wave are NF * 8 gate rows and the up rows of the same output columns
  auto w_row = [&](const RingTile& t, int c) __attribute__((always_inline)) {
    constexpr int kHalf = NF * 8;
    const int strip = c / (2 * kHalf), r = c - strip * 2 * kHalf;
    return r < kHalf ? t.n0 + strip * kHalf + r : p.act_cols + t.n0 + strip * kHalf + r - kHalf;
  };
  const bool gather = MODE == kContigListAct && p.a_rows != nullptr;
  const uint8_t *a_base, *b_base, *sp;
  uint32_t a_bytes, b_bytes, f_off;  // f_off: byte offset of the K block to fetch next
  uint32_t a_off[Cfg::A_INST], b_off[Cfg::B_INST], s_off;
  const bool fetches_as = wave < Cfg::S_WAVES;
  const int64_t sp_step = fetches_as ? p.as_sk * 4 : 4;
  // source rows of a gathered tile: from memory for the first tile, from LDS for one that was announced
  auto point_at = [&](const RingTile& t, int kb_first, bool announced) __attribute__((always_inline)) {
    int nl = lane;
    asm volatile("" : "+v"(nl));  // what is computed here is not kept in registers across the K loop
    const int r8 = nl >> 3;
    const uint32_t chunk = static_cast<uint32_t>(((nl & 7) ^ ring_swizzle(8 * wave + r8)) * 16);
    const int rows = min(BM, t.m_end - t.m0), cols = kAct ? BN : min(BN, p.N - t.n0);
    const uint32_t k0 = static_cast<uint32_t>(kb_first) * kScaleBlock;
    a_base = p.a + static_cast<int64_t>(kMaskedLike ? t.g : 0) * p.a_gs + (gather ? 0 : static_cast<int64_t>(t.m0) * p.K) + k0;
    b_base = p.b + static_cast<int64_t>(t.g) * p.b_gs + (kAct ? 0 : static_cast<int64_t>(t.n0) * p.K) + k0;
    a_bytes = (gather ? static_cast<uint32_t>(p.a_src_rows) : static_cast<uint32_t>(rows)) * uK - k0;
    b_bytes = (kAct ? static_cast<uint32_t>(p.N) : static_cast<uint32_t>(cols)) * uK - k0;
#pragma unroll
    for (int j = 0; j < Cfg::A_INST; ++j) {
      const int r = a_row(j) + r8;
      if (gather) {
        const int src = announced ? *reinterpret_cast<const int32_t*>(smem + Cfg::ROWS_OFF + r * 4) : p.a_rows[t.m0 + min(r, rows - 1)];
        a_off[j] = static_cast<uint32_t>(max(src, 0)) * uK + chunk;
      } else {
        a_off[j] = static_cast<uint32_t>(r) * uK + chunk;
      }
    }
#pragma unroll
    for (int j = 0; j < Cfg::B_INST; ++j) {
      const int r = b_row(j) + r8;
      b_off[j] = static_cast<uint32_t>(kAct ? w_row(t, r) : r) * uK + chunk;
    }
    // scales: waves below S_WAVES fetch those of 64 tile rows each, the others the weights' (lane i: of the tile's columns 32 i ..)
    const float* as_tile = p.a_s + static_cast<int64_t>(kMaskedLike ? t.g : 0) * p.as_gs + static_cast<int64_t>(t.m0) * p.as_sm + static_cast<int64_t>(kb_first) * p.as_sk;
    const float* bs_tile = p.b_s + static_cast<int64_t>(t.g) * p.bs_gs + kb_first;
    sp = reinterpret_cast<const uint8_t*>(fetches_as ? as_tile : bs_tile);
    const int c = (nl % (BN / 32)) * 32;
    const uint32_t bs_off = static_cast<uint32_t>(min((kAct ? w_row(t, c) : t.n0 + c) / kScaleBlock, p.nblocks - 1)) * static_cast<uint32_t>(p.kblocks) * 4u;
    s_off = fetches_as ? static_cast<uint32_t>(min(wave * 64 + nl, rows - 1)) * static_cast<uint32_t>(p.as_sm) * 4u : bs_off;
    f_off = 0;
  };
  // instruction i of a K step's group into stage `stage_base`: i < P1 the first part, else the second
  auto issue_one = [&](auto idx, int stage_base, uint32_t off) __attribute__((always_inline)) {
    constexpr int i = decltype(idx)::value;
    const lds_bytes_t sbase = lds + stage_base;
    constexpr bool kScale = i == Cfg::P1 - 1;
    constexpr bool kHeld = i < Cfg::H_INST;
    constexpr int j = kHeld ? i : i < Cfg::P1 - 1 ? i - Cfg::H_INST : i - Cfg::H_INST - 1;
    if constexpr (kScale) {
      uint32_t o = s_off;
      asm volatile("" : "+v"(o));
      dma_4(sp, o, sbase + (fetches_as ? Cfg::AS_OFF + wave * 256 : Cfg::WS_OFF));
    } else if constexpr (kHeld == Cfg::HOLD_X) {
      buf_dma_16<kDmaKeep>(make_rsrc(a_base, a_bytes), a_off[j], off, sbase + a_row(j) * kScaleBlock);
    } else {
      buf_dma_16<kWeightPolicy>(make_rsrc(b_base, b_bytes), b_off[j], off, sbase + Cfg::A_BYTES + b_row(j) * kScaleBlock);
    }
  };
  // slot in which instruction i of a group is issued
  constexpr auto slot_of = [](int i) {
    if (Cfg::ONE_POINT) return Cfg::B1 + 1 + i * (Cfg::T - Cfg::B1 - 1) / L;
    const int first2 = Cfg::B2 + 1 > Cfg::B1 + 1 + 2 * Cfg::P1 ? Cfg::B2 + 1 : Cfg::B1 + 1 + 2 * Cfg::P1;
    return i < Cfg::P1 ? Cfg::B1 + 1 + 2 * i : first2 + 2 * (i - Cfg::P1);
  };
  constexpr auto issued_before = [slot_of](int slot) {
    int c = 0;
    for (int i = 0; i < Cfg::P1; ++i) c += slot_of(i) < slot;
    return c;
  };
  static_assert(slot_of(L - 1) < Cfg::T, "a group is issued within its K step");

  // scale table [BM][p.sct_pitch] behind the ring: entry (r, j) = a_s of tile row r at the unit's j-th K block; lanes along K.
  auto issue_table = [&](const RingTile& t, int kb_first, int nk) __attribute__((always_inline)) {
    const int pitch = p.sct_pitch;
    const float inv_pitch = 1.0f / static_cast<float>(pitch);
    const float* as_tile = p.a_s + static_cast<int64_t>(kMaskedLike ? t.g : 0) * p.as_gs + static_cast<int64_t>(t.m0) * p.as_sm + static_cast<int64_t>(kb_first) * p.as_sk;
    const int last = min(BM, t.m_end - t.m0) - 1;
    const int n_inst = (BM * pitch + 63) >> 6;
    for (int i = wave; i < n_inst; i += Cfg::WAVES) {
      const int e = i * 64 + lane;
      const int row = static_cast<int>((static_cast<float>(e) + 0.5f) * inv_pitch);  // e / pitch, exact for e < 2^20
      const uint32_t r = static_cast<uint32_t>(min(row, last));
      const uint32_t j = static_cast<uint32_t>(min(e - row * pitch, nk - 1));
      dma_4(reinterpret_cast<const uint8_t*>(as_tile), (r * static_cast<uint32_t>(p.as_sm) + j * static_cast<uint32_t>(p.as_sk)) * 4u,
            lds + Cfg::SCTAB_OFF + i * 256);
    }
  };

  // ---- LDS reads --------------------------------------------------------------------------------------------
  // A lane's two chunks of a row.  The matrix instruction adds the four lane groups' first chunks, then their second ones; with this
  // assignment (0 4, 2 6, 1 5, 3 7) that is the order of two chained 32 x 32 x 64 on the chunks as the other kernels read them, and
  // the only one of the 40320 that gives their bits on codes of every magnitude.
  const int chunk0 = (q & 1) * 2 + (q >> 1);
  const int frag0 = ring_row(0, l16) * kScaleBlock + ((chunk0 ^ ring_swizzle(ring_row(0, l16))) << 4);
  const int x0 = wm0 * kScaleBlock + frag0, w0 = Cfg::A_BYTES + wn0 * kScaleBlock + frag0;
  const int held0 = Cfg::HOLD_X ? x0 : w0, strm0 = Cfg::HOLD_X ? w0 : x0;
  // the 32 operand bytes of this lane for fragment f: its row's chunks chunk0 and chunk0 + 4
  auto read_frag = [&](int base, int f) __attribute__((always_inline)) {
    const int o = (f >> 1) * (32 * kScaleBlock) + (f & 1) * (4 * kScaleBlock);
    const v4i lo = *reinterpret_cast<const v4i*>(smem + base + o);
    const v4i hi = *reinterpret_cast<const v4i*>(smem + (base ^ 64) + o);
    return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };
  const int tile_row = ring_row(0, l16);  // tile row of fragment 0 (of the wave) this lane's results and activation scales belong to
  float sa[MF], sb[NS];
  auto read_scales = [&](int stage_base, int kbl) __attribute__((always_inline)) {
#pragma unroll
    for (int j = 0; j < NS; ++j)
      sb[j] = *reinterpret_cast<const float*>(smem + stage_base + Cfg::WS_OFF + (wn0 / 32 + (kAct ? j * (NF / 4) : j)) * 4);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      const int row = wm0 + ring_row(mi, 0) + tile_row;
      sa[mi] = Cfg::SCTAB ? *reinterpret_cast<const float*>(smem + Cfg::SCTAB_OFF + (row * p.sct_pitch + kbl) * 4)
                          : *reinterpret_cast<const float*>(smem + stage_base + Cfg::AS_OFF + row * 4);
    }
  };

  int stage = 0;        // byte offset of the stage of the current K step
  bool staged = false;  // AHEAD: the ring holds the tile's first blocks, landed or on their way
  RingTile t, tn;
  bool have = find(vb_first, t);
  for (int vb = vb_first; have; vb += gridDim.x) {
    const bool more = find(vb + static_cast<int>(gridDim.x), tn);
    if (MODE == kContiguous && (t.g < 0 || t.g >= p.G)) {
      t = tn, have = more;
      continue;
    }
    const bool sliced = MODE == kDense && !AHEAD && !ODD && p.splitk > 1;  // (launches of K slices use the kernels without AHEAD)
    const int kb_first = sliced ? t.split * p.kb_per_split : 0;  // the host leaves no slice empty
    const int nk = sliced ? min(p.kblocks, kb_first + p.kb_per_split) - kb_first : p.kblocks;  // K blocks of this unit
    // (the table of gathered rows is waited for together with the first group of the tile)
    const bool ahead = AHEAD && more && nk >= (MODE == kContigListAct ? 2 : 1) * STAGES;

    int f_left;  // K blocks of the tile being fetched that are still to be fetched
    if (AHEAD && staged) {
      f_left = nk - STAGES;
      if (Cfg::SCTAB) ring_barrier();  // the scale table has landed
    } else {
      stage = 0;
      point_at(t, kb_first, false);
      __syncthreads();  // the previous tile's readers and DMA groups are done with the ring
      if constexpr (Cfg::SCTAB) issue_table(t, kb_first, nk);
      f_left = nk;
#pragma unroll
      for (int s = 0; s < STAGES; ++s) {
        each_index([&](auto i) __attribute__((always_inline)) { issue_one(i, s * Cfg::STAGE_BYTES, f_off); }, std::make_integer_sequence<int, L>{});
        f_left = max(f_left - 1, 0);
        if (f_left > 0)
          f_off += kScaleBlock, sp += sp_step;
        else
          a_bytes = b_bytes = 0;  // past the end of K (of a tile shorter than the ring): zeros, no traffic
      }
      wait_vmcnt<(STAGES - 1) * L>();
      ring_barrier();
    }
    if (AHEAD && gather && ahead && wave < BM / 64) {
      // the next tile's source rows, on their way before any group that is waited for
      const int r = wave * 64 + lane;
      dma_4(reinterpret_cast<const uint8_t*>(p.a_rows + tn.m0), static_cast<uint32_t>(min(r, min(BM, tn.m_end - tn.m0) - 1)) * 4u, lds + Cfg::ROWS_OFF + wave * 256);
    }
    // K steps of this tile whose blocks landed before the last tile's results were stored: nothing to wait for
    const int landed = AHEAD && staged ? STAGES : 0;
    staged = ahead;

    v4f acc[MF][NF], part[4];
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int ni = 0; ni < NF; ++ni) acc[mi][ni] = v4f{0.f, 0.f, 0.f, 0.f};
#pragma unroll
    for (int i = 0; i < 4; ++i) part[i] = v4f{0.f, 0.f, 0.f, 0.f};
    v8i held[H], strm[Cfg::NB];
    float sc[MF][NS], sc_last[2] = {0.f, 0.f};
#pragma unroll
    for (int i = 0; i < H; ++i) held[i] = read_frag(held0 + stage, i);
#pragma unroll
    for (int i = 0; i < Cfg::PD; ++i) strm[i] = read_frag(strm0 + stage, i);
    read_scales(stage, 0);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int j = 0; j < NS; ++j) sc[mi][j] = sa[mi] * sb[j];

    // ---- K loop -----------------------------------------------------------------------------------------------
    // Slot s multiplies streamed fragment s / H with held fragment s % H; its scale FMAs follow two slots later.  Every step is the
    // same code.  A streamed fragment is read PD fragments ahead, the held ones are reloaded behind their last MFMA.
    // Waits: groups are issued in order, a part's is out when no more than the groups issued behind it are.
    // the fragments of a step's last two slots, whose scale FMAs belong to the next step
    constexpr int kLast0M = Cfg::HOLD_X ? H - 2 : S - 1, kLast0N = Cfg::HOLD_X ? S - 1 : H - 2;
    constexpr int kLast1M = Cfg::HOLD_X ? H - 1 : S - 1, kLast1N = Cfg::HOLD_X ? S - 1 : H - 1;
    for (int kb = 0; kb < nk; ++kb) {
      const int next = stage == (STAGES - 1) * Cfg::STAGE_BYTES ? 0 : stage + Cfg::STAGE_BYTES;
      if (f_left == 0) {
        if (ahead)
          point_at(tn, 0, true), f_left = nk;
        else
          a_bytes = b_bytes = 0;
      }
      float sc_next[MF][NS];
      const int cur_s = strm0 + stage, nxt_s = strm0 + next, nxt_h = held0 + next;
      each_index([&](auto si) __attribute__((always_inline)) {
        constexpr int s = decltype(si)::value;
        constexpr int n = s / H, m = s % H;
        if constexpr (s == Cfg::B1 || s == Cfg::B2) ring_barrier();
        each_index([&](auto ii) __attribute__((always_inline)) {
          if constexpr (slot_of(decltype(ii)::value) == s) issue_one(ii, stage, f_off);
        }, std::make_integer_sequence<int, L>{});
        // the fences pin the order MFMA -> reads -> scale FMAs
        __builtin_amdgcn_sched_barrier(0);
        if constexpr (Cfg::HOLD_X)
          part[s & 3] = mfma_16x16x128_e4m3(strm[n % Cfg::NB], held[m], v4f{0.f, 0.f, 0.f, 0.f});
        else
          part[s & 3] = mfma_16x16x128_e4m3(held[m], strm[n % Cfg::NB], v4f{0.f, 0.f, 0.f, 0.f});
        __builtin_amdgcn_sched_barrier(0);
        // a slot ahead of the hand-overs, where the branch passes under an MFMA (right at the barrier it costs 2.5 % of a long K)
        if constexpr (s == Cfg::B2 - 1) {  // the next block's first part has landed (all of it, with one hand-over)
          constexpr int kOut = Cfg::P2 + (STAGES - 2) * L + issued_before(Cfg::B2);
          if constexpr (AHEAD)
            wait_vmcnt_unless<kOut, 1>(landed - kb);
          else
            wait_vmcnt<kOut>();
          __builtin_amdgcn_sched_barrier(0);
        } else if constexpr (s == Cfg::B1 - 1) {  // this block's second part has landed
          if constexpr (AHEAD)
            wait_vmcnt_unless<(STAGES - 1) * L, 0>(landed - kb);
          else
            wait_vmcnt<(STAGES - 1) * L>();
          __builtin_amdgcn_sched_barrier(0);
        }
        if constexpr (s == Cfg::T - H) {  // the scales have been read by now; ahead of the last reads, so that nothing waits for those
#pragma unroll
          for (int i = 0; i < MF; ++i)
#pragma unroll
            for (int j = 0; j < NS; ++j) sc_next[i][j] = sa[i] * sb[j];
          __builtin_amdgcn_sched_barrier(0);
        }
        // a fragment of the second part must not be read before B1
        constexpr bool kLate = n == 0 && n + Cfg::PD >= Cfg::LOW && n + Cfg::PD < S;
        if constexpr (m == (kLate ? Cfg::B1 : 0)) {
          constexpr int f = n + Cfg::PD;
          strm[f % Cfg::NB] = f < S ? read_frag(cur_s, f) : read_frag(nxt_s, f - S);
        }
        if constexpr (n == S - 1) held[m] = read_frag(nxt_h, m);
        if constexpr (s == Cfg::B2 + 3) read_scales(next, min(kb + 1, nk - 1));
        __builtin_amdgcn_sched_barrier(0);
        constexpr int ps = (s + Cfg::T - 2) % Cfg::T, pn = ps / H, pm = ps % H;
        constexpr int pmi = Cfg::HOLD_X ? pm : pn, pni = Cfg::HOLD_X ? pn : pm;
        if constexpr (s < 2)
          acc[pmi][pni] += part[ps & 3] * sc_last[s];
        else
          acc[pmi][pni] += part[ps & 3] * sc[pmi][ns_of(pni)];
        __builtin_amdgcn_sched_barrier(0);
      }, std::make_integer_sequence<int, Cfg::T>{});
      sc_last[0] = sc[kLast0M][ns_of(kLast0N)];
      sc_last[1] = sc[kLast1M][ns_of(kLast1N)];
#pragma unroll
      for (int i = 0; i < MF; ++i)
#pragma unroll
        for (int j = 0; j < NS; ++j) sc[i][j] = sc_next[i][j];
      f_left = max(f_left - 1, 0);
      if (f_left > 0) f_off += kScaleBlock, sp += sp_step;
      stage = next;
    }
    acc[kLast0M][kLast0N] += part[(Cfg::T - 2) & 3] * sc_last[0];
    acc[kLast1M][kLast1N] += part[(Cfg::T - 1) & 3] * sc_last[1];
    if (AHEAD && Cfg::SCTAB && ahead) issue_table(tn, 0, nk);  // every wave has read the scales of the last K block

    // ---- results ----------------------------------------------------------------------------------------------
    // lane holds c[m0 + wm0 + ring_row(mi, l16)][n0 + wn0 + 32 np + 8 q + 0 .. 7] in acc[mi][2 np] and acc[mi][2 np + 1]
    int el = lane;
    asm volatile("" : "+v"(el));  // addresses of the epilogue stay out of the K loop
    const int e_row = wm0 + ring_row(0, el & 15), eq = el >> 4;
    char* c_base = static_cast<char*>(p.c);
    if (kMaskedLike && !kAct) c_base += static_cast<int64_t>(t.g) * p.c_gs * (p.out_f32 ? 4 : 2);
    // The ring runs on: its groups land before the stores go out.  The memory counter is one for loads and stores, and a
    // load behind stores is only known to have landed when they have.
    if (AHEAD && ahead) wait_vmcnt<0>();
    if constexpr (kAct) {
      // silu(gate) * up of bf16-rounded products, rounded to bf16, and the 1 x 128 quantiser, as the separate kernels apply them
      // (moe_activation.h, fp8_quant.h).  A lane has gate and up of the same columns; a row's largest magnitude is that of
      // its four lanes and of the wave columns' shares in LDS.
      float* amax_tab = reinterpret_cast<float*>(smem + Cfg::AMAX_OFF);
      uint8_t* q_out = static_cast<uint8_t*>(p.c);
      float* s_out = p.act_s;
      if (kMaskedLike) {
        q_out += static_cast<int64_t>(t.g) * p.M * p.act_q_stride;
        s_out += static_cast<int64_t>(t.g) * p.act_s_gs;
      }
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        float amax = 0.f;
#pragma unroll
        for (int ni = 0; ni < NF / 2; ++ni)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const float g0 = static_cast<float>(static_cast<__bf16>(acc[mi][ni][u])), u0 = static_cast<float>(static_cast<__bf16>(acc[mi][NF / 2 + ni][u]));
            // the masked activation rounds silu(gate) before the product (moe.py:256-257)
            const float v = kMaskedLike ? static_cast<float>(static_cast<__bf16>(u0 * static_cast<float>(static_cast<__bf16>(act_silu_f32(g0)))))
                                        : static_cast<float>(static_cast<__bf16>(act_silu_f32(g0) * u0));
            acc[mi][ni][u] = v;
            amax = fmaxf(amax, fabsf(v));
          }
        amax = fmaxf(amax, __shfl_xor(amax, 16));
        amax = fmaxf(amax, __shfl_xor(amax, 32));
        if (eq == 0) amax_tab[(e_row + ring_row(mi, 0)) * Cfg::WGN + wave % Cfg::WGN] = amax;
      }
      ring_barrier();
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        const int row = e_row + ring_row(mi, 0);
        float amax = 0.f;
#pragma unroll
        for (int w = 0; w < Cfg::WGN; ++w) amax = fmaxf(amax, amax_tab[row * Cfg::WGN + w]);
        const float scale = fmaxf(amax, p.act_eps) / 448.0f;
        const float inv_scale = 1.0f / scale;
        const int m = t.m0 + row;
        const bool live = m < t.m_end;
        uint8_t* q_row = q_out + static_cast<int64_t>(m) * p.act_q_stride + t.n0 + wn0 / 2 + eq * 8;
#pragma unroll
        for (int np = 0; np < NF / 4; ++np) {
          int packed[2];
#pragma unroll
          for (int f = 0; f < 2; ++f) {
            float c4[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) c4[u] = fminf(fmaxf(act_div_by_scale(acc[mi][2 * np + f][u], scale, inv_scale), -448.0f), 448.0f);
            int wd = __builtin_amdgcn_cvt_pk_fp8_f32(c4[0], c4[1], 0, false);
            packed[f] = __builtin_amdgcn_cvt_pk_fp8_f32(c4[2], c4[3], wd, true);
          }
          if (live) *reinterpret_cast<v2i*>(q_row + np * 32) = v2i{packed[0], packed[1]};
        }
        if (live && eq == 0 && wave % Cfg::WGN == 0) s_out[static_cast<int64_t>(m) * p.act_s_sm + static_cast<int64_t>(t.n0 / kScaleBlock) * p.act_s_sk] = scale;
      }
    } else if (!ODD && sliced && p.fused_reduce) {
      // Split-K in one launch.  The workgroups of a tile (one per K slice) park their fp32 sums in the workspace,
      // count themselves in on the tile's arrival counter, wait - for a bounded time - until all slices are in, and
      // then each adds up its share of the tile: the slices in index order (the same order, and so the same bits, as
      // fp8_splitk_reduce_kernel), cast, store.  Nobody depends on that wait for correctness: a workgroup that gives
      // up sets its bit in the tile's word of abandoned shares and looks at the counter once more (all in after all:
      // it adds its share anyway); the workgroup whose arrival completed the tile reads that word after its own share
      // and adds the shares named there.  A share that both of them add is stored twice with the same bits.  The last
      // workgroup to leave the tile zeroes its three counters: the workspace head is all zero when the launch ends.
      // Partial sums are written in accumulator order: unit (wave MF + mi) NF + ni holds, for lane l, its four floats of that fragment.
      constexpr int kTileFloats = BM * BN;
      constexpr int kUnits = kTileFloats / 4;
      const int slices = p.splitk;
      float* tbase = p.ws + static_cast<int64_t>(t.lin) * slices * kTileFloats;
      float* mine = tbase + static_cast<int64_t>(t.split) * kTileFloats;
#pragma unroll
      for (int mi = 0; mi < MF; ++mi)
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) coherent_store16(mine + (((wave * MF + mi) * NF + ni) * 64 + lane) * 4, acc[mi][ni]);
      // The stores above are write-through, device-scope stores: once the memory counter has drained they are where
      // every XCD reads them.  (A release fence here would also write back the whole L2 of this XCD, once per
      // workgroup: measured at 4 - 11 us per launch.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // ... those of every wave; the ring is idle from here on
      uint32_t* ctr = p.ctr + static_cast<int64_t>(t.lin) * 4;
      volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(smem);
      const uint32_t uS = static_cast<uint32_t>(slices);
      if (tid == 0) {
        // the arrival and the first look at the counter travel together: one round trip instead of two
        const uint32_t ticket = __hip_atomic_fetch_add(ctr, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        uint32_t seen = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        const bool last = ticket + 1u == uS;
        bool all_in = last || seen >= uS;
#pragma unroll 1
        for (int spin = 0; !all_in && spin < p.spin_limit; ++spin) {
          __builtin_amdgcn_s_sleep(2);
          all_in = __hip_atomic_load(ctr, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) >= uS;
        }
        if (!all_in) {
          __hip_atomic_fetch_or(ctr + 1, 1u << t.split, __ATOMIC_SEQ_CST, __HIP_MEMORY_SCOPE_AGENT);
          all_in = __hip_atomic_load(ctr, __ATOMIC_SEQ_CST, __HIP_MEMORY_SCOPE_AGENT) >= uS;
        }
        flag[0] = all_in ? 1u << t.split : 0u;
        flag[1] = last ? 1u : 0u;
      }
      __syncthreads();
      const bool last = flag[1] != 0;
      const int64_t esz_c = p.out_f32 ? 4 : 2;
      auto add_unit = [&](int u, const v4f& sum) {
        const int ul = u & 63, f = u >> 6;  // f = (wave MF + mi) NF + ni
        const int fni = f % NF, fmi = (f / NF) % MF, fw = f / (NF * MF);
        const int m = t.m0 + (fw / Cfg::WGN) * (MF * 16) + ring_row(fmi, ul & 15);
        const int n = t.n0 + (fw % Cfg::WGN) * (NF * 16) + ring_row(fni, 4 * (ul >> 4));
        if (m >= t.m_end) return;
        char* c_row = c_base + static_cast<int64_t>(m) * p.N * esz_c;
        if (p.out_f32)
          store_row4<true>(c_row, n, sum, p.N - n);
        else
          store_row4<false>(c_row, n, sum, p.N - n);
      };
      for (int round = 0; round < (last ? 2 : 1); ++round) {
        if (round == 1) {
          // the arrival that completed the tile, done with its own share: the shares their owners gave up on
          __syncthreads();
          if (tid == 0) flag[0] = __hip_atomic_load(ctr + 1, __ATOMIC_SEQ_CST, __HIP_MEMORY_SCOPE_AGENT);
          __syncthreads();
        }
        const uint32_t todo = flag[0];
        for (int j = 0; j < slices; ++j) {
          if (!((todo >> j) & 1u)) continue;
          const int u0 = static_cast<int>(static_cast<int64_t>(j) * kUnits / slices);
          const int u1 = static_cast<int>(static_cast<int64_t>(j + 1) * kUnits / slices);
          // two units per thread and pass, the loads of up to eight slices of both in flight before the first sum
          for (int ua = u0 + tid; ua < u1; ua += 2 * Cfg::NT) {
            const int ub = ua + Cfg::NT;
            const bool has_b = ub < u1;
            v4f sum_a = {0.f, 0.f, 0.f, 0.f}, sum_b = {0.f, 0.f, 0.f, 0.f};
            for (int first = 0; first < slices; first += 8) {
              v4f pa[8], pb[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                pa[i] = pb[i] = v4f{0.f, 0.f, 0.f, 0.f};
                if (first + i < slices) {
                  pa[i] = coherent_load16(tbase + static_cast<int64_t>(first + i) * kTileFloats + ua * 4);
                  if (has_b) pb[i] = coherent_load16(tbase + static_cast<int64_t>(first + i) * kTileFloats + ub * 4);
                }
              }
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (first + i < slices) sum_a += pa[i], sum_b += pb[i];
            }
            add_unit(ua, sum_a);
            if (has_b) add_unit(ub, sum_b);
          }
        }
      }
      __syncthreads();  // flag[] is read; the next tile may use the ring
      if (tid == 0) {
        const uint32_t left = __hip_atomic_fetch_add(ctr + 2, 1u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        if (left + 1u == uS) {
          __hip_atomic_store(ctr, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(ctr + 1, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
          __hip_atomic_store(ctr + 2, 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        }
      }
    } else {
      // fp32 also for the first pass of split-K: the slice's sums as an [M][N] matrix of their own in the workspace, which
      // fp8_splitk_reduce_kernel, launched behind this kernel on the same stream, adds in index order
      const bool cols_inside = t.n0 + wn0 + NF * 16 <= p.N;  // no column of the wave's tile lies past N: stores without a tail
      // The four lanes of consecutive rows exchange chunks first, so that an instruction writes 256 bytes (128 in narrower wave tiles) of a
      // row instead of 64, or of 16-byte pieces of fp32.  us per call, both on one GPU: bf16 rows at odd addresses 914 x 28119 x 512 38.8 ->
      // 32.4, 3779 x 6111 x 1024 45.4 -> 36.3, 2000 x 5001 x 4096 52.0 -> 47.6; fp32 914 x 28120 x 512 39.3 -> 32.1, 271 x 18112 x 640 13.9 ->
      // 12.0; bf16 rows on 16 bytes 271 x 18112 x 640 11.1 -> 10.1, 3500 x 4096 x 512 15.1 -> 14.2, 4096 x 24576 x 1536 141 -> 138.
      // Neighbouring lanes then hold chunks 64 bytes apart, which is as good as any order where rows lie on dwords.  ODD: elsewhere the lanes
      // of a row's chunks exchange first, so that neighbours write 64 bytes (32 in narrower wave tiles) on end.  In kernels of its own,
      // because beside this form other calls lose up to 1 %.
      auto store_tile = [&](auto f32, auto inside, void* out) __attribute__((always_inline)) {
        constexpr bool F32 = decltype(f32)::value, FAR = ODD && !F32;
        const int col = t.n0 + wn0 + (FAR ? 0 : eq * 8);
#pragma unroll
        for (int mi = 0; mi < MF; ++mi) {
          // chunk `at` columns behind col, of row r of the lane's four
          auto put = [&](int r, int at, v4i v) __attribute__((always_inline)) {
            const int m = t.m0 + e_row - (el & 3) + r + ring_row(mi, 0);
            if (m >= t.m_end) return;
            char* dst = static_cast<char*>(out) + (static_cast<int64_t>(m) * p.N + col) * (F32 ? 4 : 2);
            const int n_left = p.N - col - at;
            if constexpr (F32)
              store_row4<true>(dst, at, __builtin_bit_cast(v4f, v), inside ? 4 : n_left);
            else if (inside || n_left > 0)
              store_row8_bf16(reinterpret_cast<__bf16*>(dst) + at, v, inside ? 8 : n_left);
          };
          constexpr int CHUNKS = F32 ? NF : NF / 2, kFour = CHUNKS / 4 * 4;
          auto chunk = [&](int c) __attribute__((always_inline)) {
            if constexpr (F32) {
              return __builtin_bit_cast(v4i, acc[mi][c]);
            } else {
              const v4bf lo = __builtin_convertvector(acc[mi][2 * c], v4bf), hi = __builtin_convertvector(acc[mi][2 * c + 1], v4bf);
              const v2i a = __builtin_bit_cast(v2i, lo), b = __builtin_bit_cast(v2i, hi);
              return v4i{a.x, a.y, b.x, b.y};
            }
          };
          auto chunk_col = [](int c) __attribute__((always_inline)) { return F32 ? (c >> 1) * 32 + (c & 1) * 4 : c * 32; };
          const int j = el & 3;
#pragma unroll
          for (int c = 0; c < kFour; c += 4) {
            v4i x[4] = {chunk(c), chunk(c + 1), chunk(c + 2), chunk(c + 3)};
            if constexpr (FAR) {
              swap_far_chunks<16>(x[0], x[1]), swap_far_chunks<16>(x[2], x[3]);
              swap_far_chunks<32>(x[0], x[2]), swap_far_chunks<32>(x[1], x[3]);
            }
            swap_chunks<1>(x[0], x[1], el), swap_chunks<1>(x[2], x[3], el);
            swap_chunks<2>(x[0], x[2], el), swap_chunks<2>(x[1], x[3], el);
#pragma unroll
            for (int r = 0; r < 4; ++r) put(r, FAR ? chunk_col(c + eq) + 8 * j : chunk_col(c) + chunk_col(j), x[r]);
          }
#pragma unroll
          for (int c = kFour; c + 1 < CHUNKS; c += 2) {
            v4i x[2] = {chunk(c), chunk(c + 1)};
            if constexpr (FAR) swap_far_chunks<16>(x[0], x[1]);
            swap_chunks<1>(x[0], x[1], el);
#pragma unroll
            for (int r = 0; r < 2; ++r) put((j & 2) + r, FAR ? chunk_col(c + (eq & 1)) + (eq & 2) * 8 + 8 * (j & 1) : chunk_col(c) + chunk_col(j & 1), x[r]);
          }
          if constexpr (CHUNKS % 2 != 0) put(j, chunk_col(CHUNKS - 1) + (FAR ? eq * 8 : 0), chunk(CHUNKS - 1));
        }
      };
      void* out = sliced ? static_cast<void*>(p.ws + static_cast<int64_t>(t.split) * p.M * p.N) : static_cast<void*>(c_base);
      constexpr std::true_type yes{};
      constexpr std::false_type no{};
      if (!ODD && (sliced || p.out_f32))
        cols_inside ? store_tile(yes, yes, out) : store_tile(yes, no, out);
      else
        cols_inside ? store_tile(no, yes, out) : store_tile(no, no, out);
    }
    if (!AHEAD || !ahead) wait_vmcnt<0>();  // the empty groups behind the end of K must not land in the next tile's ring
    t = tn, have = more;
  }
}

template <class Cfg, int MODE, bool AHEAD, bool ODD>
__global__ void __launch_bounds__(Cfg::NT) fp8_gemm_ring_kernel(const Args p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  ring_body<Cfg, MODE, AHEAD, ODD>(p, smem, blockIdx.x, p.tiles_m, p.tiles_n, 0);
}

// Dense GEMM whose columns are cut at p.n_split into a region of CfgA tiles and a region of narrower CfgB tiles,
// one workgroup per tile, region A first.  The host picks the cut so that the last round of workgroups fills the
// chip: e.g. 448 tiles of 256 x 256 on 256 CUs leave a quarter of the chip idle in the second round, while 256
// tiles of 256 x 256 followed by 256 tiles of 256 x 192 cover the same output and keep every CU busy.
template <class CfgA, class CfgB, bool ODD>
__global__ void __launch_bounds__(CfgA::NT) fp8_gemm_ring_mixed_kernel(const Args p) {
  static_assert(CfgA::NT == CfgB::NT && CfgA::BM == CfgB::BM, "both regions use the same workgroup shape and tile height");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int bid = blockIdx.x;
  if (bid < p.tiles_a)
    ring_body<CfgA, kDense, false, ODD>(p, smem, bid, p.tiles_m, p.tiles_n_a, 0);
  else
    ring_body<CfgB, kDense, false, ODD>(p, smem, bid - p.tiles_a, p.tiles_m, p.tiles_n_b, p.n_split);
}

// Expert-contiguous rows from the three tile lists (see contiguous_tile_list_block): persistent workgroups.  The 192-row pairs first:
// every workgroup starts at the same moment, so the two tiles of a pair run in step from their first K block (2 - 4 % over
// starting them behind the 256-row tiles); then the 256-row tiles, then the 128-row ones.
// kContigListAct: the gate/up projection of an expert MLP with the activation and the quantiser of its output in the epilogue
// (dlblas/kernels/fused_moe_v3.py:307-334 as one kernel): weights [G][2 I][K] with the gate rows first, output
// e4m3 [M][I] + scales [M][I / 128]; tiles_n = I / 128.
template <class CfgA, class CfgC, class CfgB, class CfgP, int MODE>
__global__ void __launch_bounds__(CfgA::NT) fp8_gemm_ring_list_kernel(const Args p) {
  static_assert(CfgA::NT == CfgB::NT && CfgA::NT == CfgC::NT && CfgA::NT == CfgP::NT && CfgA::BN == CfgB::BN && CfgA::BN == CfgC::BN && CfgA::BN == CfgP::BN,
                "the tile heights use the same workgroup shape and width");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int grid = static_cast<int>(gridDim.x);
  const int total_a = p.tlist[0] * p.tiles_n, total_c = p.tlist[1] * p.tiles_n, total_b = p.tlist[2] * p.tiles_n;
  // The tiles a last round would hold too few of: cut where that round then takes their 64-row pieces, one for a workgroup at most.
  // A piece's K step is bound by its 40 KB of loads, a whole tile's by its latency, so a round of pieces takes 25 to 35 us where one
  // of whole tiles takes 56 (K = 7168); two rounds of pieces are no faster than one of tiles.  us per call without / with,
  // 4096 x 7168, experts of 256 rows: 17 experts 183 / 151, 20 185 / 167, 33 286 / 270, 36 298 / 290; of 384 rows: 17 230 / 214; 14
  // of 256 and 18 of 384 rows 339 / 326.  No difference without a cut.
  const int rest = (total_a + total_b + total_c) % grid;
  const int cut_a = rest <= total_a && rest * 4 <= grid ? rest : 0, cut_c = rest > total_a && rest <= total_c && rest * 3 <= grid ? rest : 0;
  ring_body<CfgC, MODE, true>(p, smem, blockIdx.x, 0, p.tiles_n, 0, {1, 0, total_c - cut_c, 1});
  ring_body<CfgA, MODE, true>(p, smem, continue_round_robin(total_c - cut_c), 0, p.tiles_n, 0, {0, 0, total_a - cut_a, 1});
  ring_body<CfgB, MODE, true>(p, smem, continue_round_robin(total_a + total_c - cut_a - cut_c), 0, p.tiles_n, 0, {2, 0, total_b, 1});
  const ListRegion pieces = cut_a > 0 ? ListRegion{0, total_a - cut_a, cut_a, 4} : ListRegion{1, total_c - cut_c, cut_c, 3};
  ring_body<CfgP, MODE, true>(p, smem, blockIdx.x, 0, p.tiles_n, 0, pieces);
}

}  // namespace dlb
