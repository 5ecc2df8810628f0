// Weight-streaming grouped FP8 block-scaled GEMM for gfx950: experts with at most a few dozen rows each (decode steps,
// short prefill chunks), where reading every expert's weights once from HBM is the whole cost.
//
// One persistent workgroup per CU walks its tiles with ONE LDS ring that runs on across tile boundaries: the DMA of the
// next tile's first K blocks is issued STAGES steps ahead like any other, so a CU never drains its loads between two
// tiles.  What the ring needs for that:
//   - sources are addressed through buffer descriptors: a lane's byte offset (row x K + chunk) is the same for every tile,
//     only scalar registers change with the tile, and rows past an expert's last one are out of the descriptor's range
//     (the load returns zero and asks memory for nothing), so no per-tile address arithmetic sits in the issue path;
//   - the epilogue leaves from the accumulator registers and never touches the ring;
//   - activation scales go into a small double-buffered table in LDS, a chunk of K blocks at a time, by the same DMA
//     queue: no re-layout launch, one line request per row and chunk; weight scales come through scalar loads.
//
// Measured (MI355X, 32 experts, against the 128 x 256 ring kernel it replaces there): gate/up + activation 4096 x 7168,
// ~16 / ~32 rows per expert 186 -> 143 / 161 -> 148 us, down 7168 x 2048 97 -> 83 / 101 -> 91 us; 940 MB of weights at 4 rows
// 138 us = 6.8 TB/s, i.e. 12 us + bytes at 7.5 TB/s.  Where the library chooses it 1.20 x for the plain product, 1.18 x with the
// quantising epilogue (bench.py --planner-sweep stream, 70 of 96 problems of 8 .. 32 experts, up to 512 rows per expert, geometric
// means; the largest gains where 256-column tiles left CUs idle).  With AHEAD (below)
// 0 .. 256 rows: 7168 x 2048 141 -> 128 us with cold operands, 8 experts x 4096 x 7168 88 -> 68, 16 x 1024 x 2048 (0 .. 448
// rows) 37 -> 25.  Its 128 x 256 step without any load takes 0.85 us, half of that the 128 KB of fragment reads.  The longest
// experts stay with the ring kernels, whose 256-row tiles read less LDS per product.
//
// Arithmetic: fp8_gemm_kernel of the reference (dlblas/kernels/fp8_gemm.py:49-60), same order of additions as the ring
// kernels (fp8_gemm_ring.h), so results have the same bits.  Requires K % 128 == 0 and K / 128 >= STAGES.
#pragma once

#include "fp8_gemm_common.h"
#include "fp8_gemm_pipelined.h"

namespace dlb {

// What the epilogue does: store the product; silu(gate) * up + quantise with one rounding (expert-contiguous rows) or
// with the masked activation's two (dlblas/kernels/moe.py:256-257); or leave the fp32 sums of one K slice of the product, for the
// reduction kernel at the end of this file.
enum StreamEpilogue : int { kStoreProduct = 0, kSiluQuant = 1, kSiluQuantMasked = 2, kStoreSlice = 3 };

// SPLIT: as many waves again issue every load, the others only compute and store.  The loads of a step then don't wait for the stores
// of a tile, which share a wave's memory counter, and the computing waves, whose short steps are mostly issue, carry no address
// arithmetic.  Their bf16 stores write through the L2: the end of the launch has fewer lines to flush.  us per call without / with:
// 64 x 64 tiles 8 experts x 0 .. 64 rows x 1792 x 6656 29.7 / 24.3, 16 x 1024 x 2048 12.8 / 10.6, 8 x 0 .. 32 x 1024 x 4096 17.4 / 13.3;
// 64 x 128 tiles 32 x 0 .. 64 x 7168 x 2048 88.3 / 82.0, 2048 x 7168 85.5 / 79.4, 16 x 1024 x 2048 15.2 / 12.9.  The plain product in
// 256-column tiles, whose steps are long, loses where K is short (16 x 768 x 1024 10.9 / 11.8) and keeps one kind of wave; with
// the quantising epilogue it gains 1 %.  Of eight computing waves the registers leave no room for others.
template <int WGM_, int WGN_, int MF_, int NF_, int STAGES_, int CH_, bool SPLIT_ = false>
struct StreamCfg {
  static constexpr int WGM = WGM_, WGN = WGN_, MF = MF_, NF = NF_, STAGES = STAGES_;
  static constexpr int WAVES = WGM * WGN;
  static constexpr bool SPLIT = SPLIT_;
  static constexpr int NT = (SPLIT ? 2 : 1) * WAVES * 64;
  static constexpr int BM = WGM * MF * 32;
  static constexpr int BN = WGN * NF * 32;
  static constexpr int A_INST = BM / 8 / WAVES;
  static constexpr int B_INST = BN / 8 / WAVES;
  static constexpr int A_BYTES = BM * kScaleBlock;
  static constexpr int B_BYTES = BN * kScaleBlock;
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES;
  static constexpr int L = A_INST + B_INST;  // vmcnt units per wave and step, scale chunks aside
  static constexpr int CH = CH_;             // K blocks per chunk of the scale table, at most
  static constexpr int PITCH = CH | 1;       // floats per table row (odd: 32 rows lie in 32 banks)
  static constexpr int TAB_INST = (BM * PITCH + 64 * WAVES - 1) / (64 * WAVES);  // DMA instructions per wave and chunk
  static constexpr int TAB_BYTES = TAB_INST * WAVES * 256;
  static constexpr int TAB_OFF = STAGES * STAGE_BYTES;
  static constexpr int ROW_OFF = TAB_OFF + 2 * TAB_BYTES;  // source rows of the issue tile (gathered activations)
  static constexpr int MAX_OFF = ROW_OFF + BM * 4;         // row maxima of the waves (quantising epilogue)
  static constexpr int LDS_BYTES = MAX_OFF + WGN * BM * 4;
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "tile rows must divide over the DMA instructions");
  static_assert(!SPLIT || WAVES == 4, "eight waves share the registers");
  static_assert(WAVES % 2 == 0, "chunk swizzle must not depend on the DMA instruction index");
  static_assert(L * (STAGES - 1) < 64, "vmcnt is a 6-bit counter");
  static_assert(LDS_BYTES <= 160 * 1024, "ring, table and row maxima fit the LDS");
};

typedef const __attribute__((address_space(4))) float* const_float_ptr_t;
typedef unsigned v4u __attribute__((ext_vector_type(4)));

// Wait until at most `younger` (0 .. MAX) groups of L vector-memory instructions are on their way.
template <int L, int MAX>
__device__ __forceinline__ void wait_groups(int younger) {
  if constexpr (MAX > 0) {
    if (younger >= MAX)
      wait_vmcnt<MAX * L>();
    else
      wait_groups<L, MAX - 1>(younger);
  } else {
    wait_vmcnt<0>();
  }
}

// Row ranges of the experts, 64 at a time: lane i of every wave holds expert first + i.
struct ExpertWalk {
  int first, base, total;  // first expert of the window, tiles before it, tiles in it
  int row0, rows, mtiles, incl;
};

// GATHER: row r of the GEMM is row a_rows[r] of a and a_s.
// AHEAD: fragments are read one step ahead of their use, in a loop without branches while an expert's tiles are full; else
// when they are needed, by the waves that need them.  Ahead is for experts of more rows than a tile has: masked layout, 32
// experts x 0 .. 256 rows, 7168 x 2048 130 -> 116 us (128 x 256 tiles; the ring kernel 141), 16 x 0 .. 128 rows, 1024 x 3072
// 20.3 -> 19.1 us.  Short experts lose by it (8 experts, 12 rows, 3200 x 1280: 9.7 -> 10.9 us): most of their steps take the
// path with the branches.
template <class Cfg, int EPI, bool GATHER, bool AHEAD>
__global__ void __launch_bounds__(Cfg::NT) fp8_gemm_stream_kernel(const Args p) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, MF = Cfg::MF, NF = Cfg::NF, WAVES = Cfg::WAVES, WGM = Cfg::WGM, STAGES = Cfg::STAGES;
  constexpr bool kAct = EPI == kSiluQuant || EPI == kSiluQuantMasked;
  constexpr bool kSliced = EPI == kStoreSlice;
  static_assert(!kAct || BN == 256, "a quantisation group is the 128 output columns of 256 weight rows");
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  constexpr bool kSplit = Cfg::SPLIT;
  const int wave_id = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const bool loads = kSplit && wave_id >= WAVES;  // this wave issues loads and nothing else
  const int wave = loads ? wave_id - WAVES : wave_id;
  const int l32 = lane & 31, h = lane >> 5;
  const int wrow = wave / Cfg::WGN;  // the wave's fragment mi is the tile's fragment mi WGM + wrow: wave rows share short tiles evenly
  const LaneChunks lc = make_lane_chunks(l32, h);
  const int slices = kSliced ? p.splitk : 1;
  const int grid = static_cast<int>(gridDim.x);
  const int bid = static_cast<int>(blockIdx.x);
  // the row tiles of an expert are adjacent in the order; of every 32 consecutive tiles an XCD takes 4 consecutive ones
  const int slot0 = (bid / 32) * 32 + (bid % 8) * 4 + (bid / 8) % 4;

  ExpertWalk ew;
  auto load_window = [&](int first, int base) {
    ew.first = first;
    ew.base = base;
    const int e = first + lane;
    int row0 = 0, rows = 0;
    if (e < p.G) {
      if (p.row_start != nullptr) {
        row0 = p.row_start[e];
        rows = max(p.gidx[e] - row0, 0);
      } else {
        row0 = e * p.M;
        rows = min(max(p.gidx[e], 0), p.M);
      }
    }
    ew.row0 = row0;
    ew.rows = rows;
    ew.mtiles = (rows + BM - 1) / BM;
    int incl = ew.mtiles * p.tiles_n * slices;
#pragma unroll
    for (int off = 1; off < 64; off <<= 1) {
      const int up = __shfl_up(incl, off);
      if (lane >= off) incl += up;
    }
    ew.incl = incl;
    ew.total = __builtin_amdgcn_readlane(incl, 63);
  };

  // one tile: wave-uniform
  struct Tile {
    int g, row, rows, n0;  // expert, first row (of a / of the output), valid rows, first weight row / output column
    int slice, kb0, kb1;   // K slice: blocks [kb0, kb1)
    bool ok;
  };
  auto first_kb = [&](const Tile& t) __attribute__((always_inline)) { return kSliced ? t.kb0 : 0; };
  auto end_kb = [&](const Tile& t) __attribute__((always_inline)) { return kSliced ? t.kb1 : p.kblocks; };
  auto locate = [&](int id) {
    Tile t{};
    while (id >= ew.base + ew.total) {
      if (ew.first + 64 >= p.G) return t;
      load_window(ew.first + 64, ew.base + ew.total);
    }
    const int rel = id - ew.base;
    const int i = __builtin_ctzll(__ballot(ew.incl > rel));
    const int mtiles = __builtin_amdgcn_readlane(ew.mtiles, i);
    const int per_slice = mtiles * p.tiles_n;
    int local = rel - (__builtin_amdgcn_readlane(ew.incl, i) - per_slice * slices);
    if (kSliced) {
      // K slices of equal length, the first few one block longer
      const int longer = p.kblocks - slices * p.kb_per_split;
      t.slice = local / per_slice;
      local -= t.slice * per_slice;
      t.kb0 = t.slice * p.kb_per_split + min(t.slice, longer);
      t.kb1 = t.kb0 + p.kb_per_split + (t.slice < longer ? 1 : 0);
    }
    const int nt = local / mtiles, mt = local - nt * mtiles;
    t.g = ew.first + i;
    // the row tiles of an expert are equally high (in fragments): they run side by side and share its weights in the L2
    const int rows = __builtin_amdgcn_readlane(ew.rows, i);
    const int height = ((rows + 31) / 32 + mtiles - 1) / mtiles * 32;
    t.row = __builtin_amdgcn_readlane(ew.row0, i) + mt * height;
    t.rows = min(height, rows - mt * height);
    t.n0 = nt * (kAct ? BN / 2 : BN);
    t.ok = true;
    return t;
  };

  // ---- issue side --------------------------------------------------------------------------------------------------
  const int dma_row = 8 * wave + (lane >> 3);
  const uint32_t dma_chunk = static_cast<uint32_t>(((lane & 7) ^ chunk_swizzle(dma_row)) * 16);
  const uint32_t uK = static_cast<uint32_t>(p.K);
  uint32_t a_off[Cfg::A_INST], b_off[Cfg::B_INST];
#pragma unroll
  for (int j = 0; j < Cfg::A_INST; ++j) a_off[j] = static_cast<uint32_t>(dma_row + 8 * j * WAVES) * uK + dma_chunk;
#pragma unroll
  for (int j = 0; j < Cfg::B_INST; ++j) {
    const int c = dma_row + 8 * j * WAVES;
    // quantising epilogue: tile rows 0 .. 127 are gate rows, 128 .. 255 the up rows of the same output columns
    b_off[j] = static_cast<uint32_t>(kAct && c >= BN / 2 ? p.act_cols + c - BN / 2 : c) * uK + dma_chunk;
  }
  int* rows_lds = reinterpret_cast<int*>(smem + Cfg::ROW_OFF);
  // scale table: entry (row, j) of a chunk at row * tab_rs + j * tab_js; the side that is contiguous in a_s is the
  // contiguous one here too, so that a DMA instruction moves whole runs
  const bool tab_by_row = p.as_sk == 1;
  const int tab_rs = tab_by_row ? Cfg::PITCH : 1, tab_js = tab_by_row ? 1 : BM;

  Tile it;                      // the tile the issue side works on
  int it_seq = 0, it_kb = 0;    // its number in this workgroup's sequence; its next K block (counted from the first of all slices)
  int it_stage = 0, it_tab = 0, it_chunk_kb = 0;
  __amdgpu_buffer_rsrc_t a_src, b_src;
  const float* as_src = nullptr;

  auto enter_tile = [&]() {
    it = locate(it_seq * grid + slot0);
    ++it_seq;
    it_kb = it_chunk_kb = first_kb(it);
    if (!it.ok) return;
    const uint8_t* bg = p.b + static_cast<int64_t>(it.g) * p.b_gs + static_cast<int64_t>(it.n0) * p.K;
    b_src = make_rsrc(bg, static_cast<uint32_t>(kAct ? p.N - it.n0 : min(BN, p.N - it.n0)) * uK);
    if (GATHER) {
      a_src = make_rsrc(p.a, static_cast<uint32_t>(p.a_src_rows) * uK);
      as_src = p.a_s;
      // every wave fetches and writes the whole list itself (same values): no barrier
      for (int r = lane; r < BM; r += 64) rows_lds[r] = r < it.rows ? max(p.a_rows[it.row + r], 0) : -1;
#pragma unroll
      for (int j = 0; j < Cfg::A_INST; ++j) {
        const int src = rows_lds[dma_row + 8 * j * WAVES];
        a_off[j] = src < 0 ? 0x80000000u : static_cast<uint32_t>(src) * uK + dma_chunk;  // 2^31: beyond the descriptor
      }
    } else {
      a_src = make_rsrc(p.a + static_cast<int64_t>(it.row) * p.K, static_cast<uint32_t>(it.rows) * uK);
      // masked layout: a_s has a group stride of its own; t.row counts rows of all experts
      as_src = p.row_start != nullptr ? p.a_s + static_cast<int64_t>(it.row) * p.as_sm
                                      : p.a_s + static_cast<int64_t>(it.g) * p.as_gs + static_cast<int64_t>(it.row - it.g * p.M) * p.as_sm;
    }
  };

  auto issue_loads = [&]() __attribute__((always_inline)) {
    uint8_t* sbase = smem + it_stage * Cfg::STAGE_BYTES;
    const uint32_t koff = static_cast<uint32_t>(it_kb) * kScaleBlock;
#pragma unroll
    for (int j = 0; j < Cfg::B_INST; ++j) buf_dma_16<kDmaStream>(b_src, b_off[j], koff, sbase + Cfg::A_BYTES + (j * WAVES + wave) * 1024);
#pragma unroll
    for (int j = 0; j < Cfg::A_INST; ++j) buf_dma_16<kDmaKeep>(a_src, a_off[j], koff, sbase + (j * WAVES + wave) * 1024);
    ++it_kb;
    it_stage = it_stage + 1 == STAGES ? 0 : it_stage + 1;
  };
  auto open_chunk = [&]() {
    if (it_kb == it_chunk_kb) {
      // this step opens a chunk of the scale table
      const int len = min(p.chunk_len, end_kb(it) - it_kb);
      uint8_t* tab = smem + Cfg::TAB_OFF + it_tab * Cfg::TAB_BYTES;
#pragma unroll
      for (int i = 0; i < Cfg::TAB_INST; ++i) {
        const int e = (i * WAVES + wave) * 64 + lane;
        int row = tab_by_row ? static_cast<int>((static_cast<float>(e) + 0.5f) * (1.0f / Cfg::PITCH)) : e % BM;
        int j = tab_by_row ? e - row * Cfg::PITCH : e / BM;
        row = min(row, it.rows - 1);
        j = min(j, len - 1);
        if (GATHER) row = rows_lds[row];
        dma_4(reinterpret_cast<const uint8_t*>(as_src + static_cast<int64_t>(row) * p.as_sm + static_cast<int64_t>(it_kb + j) * p.as_sk), 0,
              tab + (i * WAVES + wave) * 256);
      }
      it_tab ^= 1;
      it_chunk_kb += p.chunk_len;
    }
  };
  auto issue_step = [&]() {
    if (it.ok && it_kb == end_kb(it)) enter_tile();
    if (!it.ok) return;
    open_chunk();
    issue_loads();
  };
  // kSplit, waves that compute: `it` is the tile after ct
  auto advance = [&]() { it = locate(it_seq++ * grid + slot0); };

  load_window(0, 0);
  if (kSplit && !loads)
    advance();
  else
    enter_tile();
  if (!it.ok) return;
  Tile ct = it;  // the tile the compute side works on
  if (!kSplit || loads) {
    // a tile has at least STAGES K blocks and a chunk at least STAGES - 1.  (Gathered rows in whole steps: the compiler then spills 37 to
    // 51 scalar registers there in place of 60 to 71, 16 experts x ~48 gathered rows x 3328 x 1792 21.4 -> 21.0 us.)
    if constexpr (GATHER) {
#pragma unroll
      for (int s = 0; s < STAGES - 1; ++s) issue_step();
    } else {
      open_chunk();
#pragma unroll
      for (int s = 0; s < STAGES - 1; ++s) issue_loads();
    }
    if (AHEAD) {
      open_chunk();
      issue_loads();
    }
  }
  if constexpr (kSplit) {
    if (loads) {
      // in step with the waves that compute, barrier for barrier: of step `done`, and of a tile's quantising epilogue
      if (AHEAD) {
        wait_vmcnt<(STAGES - 1) * Cfg::L>();
        lds_barrier();
      }
      int left = p.kblocks;
      for (int done = 0, issued = STAGES - 1 + (AHEAD ? 1 : 0); done < issued; ++done) {
        // (AHEAD: the next block's loads have landed; else this one's)
        wait_groups<Cfg::L, STAGES - 2>(issued - done - (AHEAD ? 2 : 1));
        lds_barrier();
        issue_step();
        if (it.ok) ++issued;
        if (kAct && --left == 0) {
          left = p.kblocks;
          lds_barrier();
        }
      }
      return;
    }
    advance();
  }

  // ---- compute side ------------------------------------------------------------------------------------------------
  // AHEAD: the fragments of a K block are in registers when its step begins; each is replaced by the next block's as soon as
  // the last matrix instruction that reads it has been issued.  Most steps open no tile and no chunk of the scale table and
  // have valid rows in every fragment: those run in a loop of their own (run_fast) without a branch; the others skip
  // fragments whose rows are all past the expert's last one, reads included.  (With the checks in every step their 150 scalar
  // instructions were the bound: 1.1 us a 128 x 256 step without any load, now 0.85.  A loop for every number of live
  // fragments made the compiler spill: 2.8 x slower.)
  const int wn0 = (wave % Cfg::WGN) * (NF * 32);
  int frag_off[NF];  // lane-dependent for the quantising epilogue
#pragma unroll
  for (int ni = 0; ni < NF; ++ni) {
    // kAct: fragment rows 0 .. 15 are the gate rows of 16 output columns, 16 .. 31 their up rows.  l32 >= 16 then reads LDS
    // row 128 + 16 f + (l32 - 16); row & 15 is the same, so the lane's swizzled chunk offsets hold
    frag_off[ni] = Cfg::A_BYTES + (kAct ? ((wave % Cfg::WGN) * NF + ni) * 16 + (l32 >= 16 ? BN / 2 - 16 : 0) : wn0 + ni * 32) * kScaleBlock;
  }
  v8i x[MF][2], w[NF][2];
  float sa[MF];
  int base = 0;                     // ring stage (in bytes) of the block whose fragments are read next
  int tab = 0;                      // its buffer of the scale table
  int tab_kb = 0, chunk_end = 0;    // its number in its chunk; the first block of the chunk after it
  const float* tab_ptr = nullptr;
  auto frag_row = [&](int mi) { return (mi * WGM + wrow) * 32; };
  auto read_x = [&](int mi) __attribute__((always_inline)) {
    x[mi][0] = lds_read_frag32(smem, base + frag_row(mi) * kScaleBlock, lc, 0);
    x[mi][1] = lds_read_frag32(smem, base + frag_row(mi) * kScaleBlock, lc, 1);
    sa[mi] = tab_ptr[(frag_row(mi) + l32) * tab_rs + tab_kb * tab_js];
  };
  auto read_w = [&](int ni) __attribute__((always_inline)) {
    w[ni][0] = lds_read_frag32(smem, base + frag_off[ni], lc, 0);
    w[ni][1] = lds_read_frag32(smem, base + frag_off[ni], lc, 1);
  };
  auto next_stage = [&]() __attribute__((always_inline)) { base = base + Cfg::STAGE_BYTES == STAGES * Cfg::STAGE_BYTES ? 0 : base + Cfg::STAGE_BYTES; };
  auto enter_block = [&](int kb, bool first) {  // block kb is the one whose fragments are read next; first: of its tile
    ++tab_kb;
    if (first) chunk_end = kb;
    if (kb == chunk_end) {
      tab_ptr = reinterpret_cast<const float*>(smem + Cfg::TAB_OFF + tab * Cfg::TAB_BYTES);
      tab ^= 1;
      tab_kb = 0;
      chunk_end += p.chunk_len;
    }
  };
  // weight scales of the wave's columns: one 128-block per wave (kAct: one for the gate, one for the up half)
  const_float_ptr_t bs0, bs1;
  auto enter_scales = [&](const Tile& t) {
    const float* bs_g = p.b_s + static_cast<int64_t>(t.g) * p.bs_gs;
    const int nb0 = kAct ? t.n0 / kScaleBlock : min((t.n0 + wn0) / kScaleBlock, p.nblocks - 1);
    bs0 = (const_float_ptr_t)(bs_g + static_cast<int64_t>(nb0) * p.kblocks);
    bs1 = (const_float_ptr_t)(bs_g + static_cast<int64_t>(kAct ? nb0 + p.act_cols / kScaleBlock : nb0) * p.kblocks);
  };
  auto multiply = [&](int ni, int mi) __attribute__((always_inline)) {
    v16f z;
#pragma unroll
    for (int u = 0; u < 16; ++u) z[u] = 0.f;
    z = mfma_32x32x64_e4m3(w[ni][0], x[mi][0], z);
    return mfma_32x32x64_e4m3(w[ni][1], x[mi][1], z);
  };
  v16f acc[MF][NF];
  float sb0, sb1;
  auto accumulate = [&](int mi, int ni, const v16f& z, float s0, float s1) __attribute__((always_inline)) {
#pragma unroll
    for (int u = 0; u < 16; ++u) acc[mi][ni][u] = fmaf(z[u], kAct && u >= 8 ? s1 : s0, acc[mi][ni][u]);
  };

  if constexpr (AHEAD) {
    enter_scales(ct);
    sb0 = bs0[first_kb(ct)], sb1 = bs1[first_kb(ct)];
    if (!kSplit) wait_vmcnt<(STAGES - 1) * Cfg::L>();
    lds_barrier();
    enter_block(first_kb(ct), true);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
      if (frag_row(mi) < ct.rows) read_x(mi);
#pragma unroll
    for (int ni = 0; ni < NF; ++ni) read_w(ni);
  }

  // n steps from block kb on: the block after each is in the same tile and chunk, and so is what each issues
  auto run_fast = [&](int kb, int n) __attribute__((always_inline)) {
    const_float_ptr_t q0 = bs0 + kb + 1, q1 = bs1 + kb + 1;
#pragma unroll 1
    for (; n > 0; --n, ++q0, ++q1) {
      v16f z[NF];
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ni = 0; ni < NF; ++ni) z[ni] = multiply(ni, 0);
      __builtin_amdgcn_sched_barrier(0);
      // the next block's loads have landed, and every wave holds this block in registers: its stage can be refilled
      if (!kSplit) wait_vmcnt<(STAGES - 2) * Cfg::L>();
      lds_barrier();
      float s0[MF], s1[MF];
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) s0[mi] = sa[mi] * sb0, s1[mi] = sa[mi] * sb1;
      sb0 = *q0;
      if (kAct) sb1 = *q1;
      else sb1 = sb0;
      if (!kSplit) issue_loads();
      next_stage();
      ++tab_kb;
      if (MF == 1) {
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) read_w(ni);
      }
      read_x(0);
      __builtin_amdgcn_sched_barrier(0);
#pragma unroll
      for (int ni = 0; ni < NF; ++ni) accumulate(0, ni, z[ni], s0[0], s1[0]);
#pragma unroll
      for (int mi = 1; mi < MF; ++mi) {
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) {
          z[ni] = multiply(ni, mi);
          if (mi == MF - 1) {
            __builtin_amdgcn_sched_barrier(0);
            read_w(ni);
            __builtin_amdgcn_sched_barrier(0);
          }
        }
        __builtin_amdgcn_sched_barrier(0);
        read_x(mi);
        __builtin_amdgcn_sched_barrier(0);
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) accumulate(mi, ni, z[ni], s0[mi], s1[mi]);
      }
    }
  };

  while (true) {
    if (!AHEAD) {
      enter_scales(ct);
      sb0 = bs0[first_kb(ct)], sb1 = bs1[first_kb(ct)];
    }
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int ni = 0; ni < NF; ++ni)
#pragma unroll
        for (int t = 0; t < 16; ++t) acc[mi][ni][t] = 0.f;
    const bool full = AHEAD && frag_row(MF - 1) < ct.rows;

    for (int kb = first_kb(ct); AHEAD && kb < end_kb(ct); ++kb) {
      if (full && (kSplit || it.ok)) {
        int n = min(end_kb(ct), chunk_end) - 1 - kb;
        if (!kSplit) n = min(n, min(end_kb(it), it_chunk_kb) - it_kb);
        if (n > 0) {
          run_fast(kb, n);
          kb += n;
        }
      }
      float s0[MF], s1[MF];
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) s0[mi] = sa[mi] * sb0, s1[mi] = sa[mi] * sb1;
      int rows_n = 0, kb_n = 0;
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        if (frag_row(mi) < ct.rows) {
          v16f z[NF];
#pragma unroll
          for (int ni = 0; ni < NF; ++ni) z[ni] = multiply(ni, mi);
#pragma unroll
          for (int ni = 0; ni < NF; ++ni) accumulate(mi, ni, z[ni], s0[mi], s1[mi]);
        }
        if (mi == 0) {
          // younger than the next block's loads: those of STAGES - 2 steps, fewer at the end of the last tile
          if (!kSplit) wait_groups<Cfg::L, STAGES - 2>(it.ok ? STAGES - 2 : end_kb(ct) - 2 - kb);
          lds_barrier();
          if (!kSplit) issue_step();
          next_stage();
          const bool next_tile = kb + 1 == end_kb(ct);
          if (!next_tile) {
            kb_n = kb + 1;
            rows_n = ct.rows;
          } else if (it.ok) {
            // the issue side is in the next tile: every tile has at least STAGES K blocks
            kb_n = first_kb(it);
            rows_n = it.rows;
            enter_scales(it);
          }
          enter_block(kb_n, next_tile);
          sb0 = bs0[kb_n];
          sb1 = bs1[kb_n];
        }
        if (frag_row(mi) < rows_n) read_x(mi);
      }
      if (frag_row(0) < rows_n) {
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) read_w(ni);
      }
    }

    if constexpr (!AHEAD) {
      for (int kb = first_kb(ct); kb < end_kb(ct); ++kb) {
        // the loads of this step have landed: behind them at most the groups of the next STAGES - 2 steps are out
        if (!kSplit) wait_groups<Cfg::L, STAGES - 2>(it.ok ? STAGES - 2 : end_kb(ct) - 1 - kb);
        lds_barrier();  // ... those of every wave, and nobody reads the stage before this one any more
        if (!kSplit) issue_step();
        enter_block(kb, kb == first_kb(ct));
        if (WGM == 1 || frag_row(0) < ct.rows) {
          v8i wf[NF][2];
#pragma unroll
          for (int ni = 0; ni < NF; ++ni) {
            wf[ni][0] = lds_read_frag32(smem, base + frag_off[ni], lc, 0);
            wf[ni][1] = lds_read_frag32(smem, base + frag_off[ni], lc, 1);
          }
#pragma unroll
          for (int mi = 0; mi < MF; ++mi) {
            if (mi > 0 && frag_row(mi) >= ct.rows) continue;  // no valid row in this fragment
            const v8i x0 = lds_read_frag32(smem, base + frag_row(mi) * kScaleBlock, lc, 0);
            const v8i x1 = lds_read_frag32(smem, base + frag_row(mi) * kScaleBlock, lc, 1);
            const float sk = tab_ptr[(frag_row(mi) + l32) * tab_rs + tab_kb * tab_js];
            const float s0 = sk * sb0, s1 = sk * sb1;
#pragma unroll
            for (int ni = 0; ni < NF; ++ni) {
              v16f z;
#pragma unroll
              for (int u = 0; u < 16; ++u) z[u] = 0.f;
              z = mfma_32x32x64_e4m3(wf[ni][0], x0, z);
              z = mfma_32x32x64_e4m3(wf[ni][1], x1, z);
              accumulate(mi, ni, z, s0, s1);
            }
          }
        }
        const int kn = min(kb + 1, end_kb(ct) - 1);
        sb0 = bs0[kn];
        sb1 = bs1[kn];
        next_stage();
      }
    }

    // ---- epilogue: lane holds rows frag_row(mi) + l32, weight rows 8 u + 4 h + 0..3 of every fragment, u = 0..3 -------
    if constexpr (kAct) {
      // u = 0, 1: gate, u = 2, 3: up of output columns c0 + 8 u + 4 h + 0..3.  The values pass through bf16 as the plain
      // GEMM would have stored them, so codes and scales have the bits of the three separate steps.
      float* maxima = reinterpret_cast<float*>(smem + Cfg::MAX_OFF);
      float amax[MF];
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        amax[mi] = 0.f;
#pragma unroll
        for (int ni = 0; ni < NF; ++ni)
#pragma unroll
          for (int t = 0; t < 8; ++t) {
            const float gate = static_cast<float>(static_cast<__bf16>(acc[mi][ni][t]));
            const float up = static_cast<float>(static_cast<__bf16>(acc[mi][ni][t + 8]));
            float v;
            if (EPI == kSiluQuantMasked)
              v = static_cast<float>(static_cast<__bf16>(up * static_cast<float>(static_cast<__bf16>(act_silu_f32(gate)))));
            else
              v = static_cast<float>(static_cast<__bf16>(act_silu_f32(gate) * up));
            acc[mi][ni][t] = v;
            amax[mi] = fmaxf(amax[mi], fabsf(v));
          }
        amax[mi] = fmaxf(amax[mi], __shfl_xor(amax[mi], 32));
        if (h == 0) maxima[(wave % Cfg::WGN) * BM + frag_row(mi) + l32] = amax[mi];
      }
      lds_barrier();
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        const int row = frag_row(mi) + l32;
#pragma unroll
        for (int w2 = 0; w2 < Cfg::WGN; ++w2) amax[mi] = fmaxf(amax[mi], maxima[w2 * BM + row]);
        const float scale = fmaxf(amax[mi], p.act_eps) / 448.0f;
        const float inv_scale = 1.0f / scale;
        // p.c / p.act_s are indexed by the row of all experts; the masked layout's scales have a group stride of their own
        uint8_t* q_row = static_cast<uint8_t*>(p.c) + static_cast<int64_t>(ct.row + row) * p.act_q_stride + ct.n0;
        const int64_t s_at = p.row_start != nullptr ? static_cast<int64_t>(ct.row + row) * p.act_s_sm
                                                    : static_cast<int64_t>(ct.g) * p.act_s_gs + static_cast<int64_t>(ct.row + row - ct.g * p.M) * p.act_s_sm;
        const bool live = row < ct.rows;
        if (live && h == 0 && wave % Cfg::WGN == 0) p.act_s[s_at + static_cast<int64_t>(ct.n0 / kScaleBlock) * p.act_s_sk] = scale;
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) {
          int packed[2];
#pragma unroll
          for (int u = 0; u < 2; ++u) {
            float c4[4];
#pragma unroll
            for (int j = 0; j < 4; ++j)
              c4[j] = fminf(fmaxf(act_div_by_scale(acc[mi][ni][4 * u + j], scale, inv_scale), -448.0f), 448.0f);
            int wd = __builtin_amdgcn_cvt_pk_fp8_f32(c4[0], c4[1], 0, false);
            packed[u] = __builtin_amdgcn_cvt_pk_fp8_f32(c4[2], c4[3], wd, true);
          }
          // lanes l and l + 32 hold columns 0-3 and 4-7 (u = 0), 8-11 and 12-15 (u = 1): after the swap the lower one has
          // columns 0-7, the upper one 8-15
          const auto sw = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(packed[0]), static_cast<unsigned>(packed[1]), false, false);
          if (live) *reinterpret_cast<v2i*>(q_row + ((wave % Cfg::WGN) * NF + ni) * 16 + 8 * h) = v2i{static_cast<int>(sw[0]), static_cast<int>(sw[1])};
        }
      }
    } else {
      // One copy of the stores per output type: with others for tiles inside the matrix the kernel spilled 60 scalar registers in
      // place of 37, and every change of tile took longer (32 experts x 0 .. 256 rows x 7168 x 2048 0.6 %).
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        const int row = frag_row(mi) + l32;
        const bool live = row < ct.rows;
        // (a K slice's sums: an [all rows][N] matrix of its own)
        const int64_t at = (kSliced ? static_cast<int64_t>(ct.slice) * p.c_gs : 0) + static_cast<int64_t>(ct.row + row) * p.N;
        char* c_row = static_cast<char*>(p.c) + at * (kSliced || p.out_f32 ? 4 : 2);
#pragma unroll
        for (int ni = 0; ni < NF; ++ni) {
          const int nf = ct.n0 + wn0 + ni * 32;
          if (!kSliced && p.c_whole) {
            // lanes l and l + 32 swap halves so that each stores 8 consecutive columns
#pragma unroll
            for (int u = 0; u < 4; u += 2) {
              v2i lo, hi;
              {
                const v4f a4 = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
                const v4f b4 = {acc[mi][ni][4 * u + 4], acc[mi][ni][4 * u + 5], acc[mi][ni][4 * u + 6], acc[mi][ni][4 * u + 7]};
                lo = __builtin_bit_cast(v2i, __builtin_convertvector(a4, v4bf));
                hi = __builtin_bit_cast(v2i, __builtin_convertvector(b4, v4bf));
              }
              const auto s0 = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(lo.x), static_cast<unsigned>(hi.x), false, false);
              const auto s1 = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(lo.y), static_cast<unsigned>(hi.y), false, false);
              const int n = nf + 8 * u + 8 * h;
              const v4i c8 = {static_cast<int>(s0[0]), static_cast<int>(s1[0]), static_cast<int>(s0[1]), static_cast<int>(s1[1])};
              if (live && n < p.N) {
                if (kSplit && p.c_whole == 2) {
                  // write-through: bit 4 of the policy is sc1
                  const __amdgpu_buffer_rsrc_t c_rsrc = make_rsrc(static_cast<const uint8_t*>(p.c) + static_cast<int64_t>(ct.row) * p.N * 2, static_cast<uint32_t>(ct.rows * p.N) * 2u);
                  __builtin_amdgcn_raw_buffer_store_b128(__builtin_bit_cast(v4u, c8), c_rsrc, static_cast<uint32_t>(row * p.N + n) * 2u, 0, 16);
                } else {
                  *reinterpret_cast<v4i_el*>(c_row + static_cast<int64_t>(n) * 2) = c8;
                }
              }
            }
          } else if (live) {
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              const int n = nf + u * 8 + h * 4;
              const v4f v = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
              if (kSliced || p.out_f32)
                store_row4<true>(c_row, n, v, p.N - n);
              else
                store_row4<false>(c_row, n, v, p.N - n);
            }
          }
        }
      }
    }
    if (!it.ok) break;  // the issue side is one tile ahead: it has found no further one
    ct = it;
    if (kSplit) advance();
  }
}

// K slices (p.splitk of them) of a gate/up projection: few experts, or narrow ones, have fewer tiles than the chip has CUs, and a CU
// fetches 40 - 50 GB/s whatever it is asked for.  The streaming kernel then runs the plain product of every (tile, K slice), fp32 sums
// in an [all rows][N] matrix per slice (p.ws, p.c_gs floats apart), and the kernel below, behind it on the stream, adds the slices in
// index order, activates and quantises: 8 experts x ~15 rows x 1792 x 3584 24.9 -> 17.0 us, 32 x ~9 rows x 512 x 5632 36.9 -> 22.4 us.
// Bound: the partial sums' way through the caches, 3 us with the launch at decode sizes; loads of up to kReduceBatch slices are in
// flight per lane.  (The plain product gains nothing from slices that smaller tiles do not give it: 1.001 x over 195 problems.)
constexpr int kReduceBatch = 4;
constexpr int kMaxStreamSlices = 8;

// rows [row0, row0 + rows) of expert g, as the streaming kernel sees them
__device__ __forceinline__ void stream_expert_rows(const Args& p, int g, int* row0, int* rows) {
  if (p.row_start != nullptr) {
    *row0 = p.row_start[g];
    *rows = max(p.gidx[g] - *row0, 0);
  } else {
    *row0 = g * p.M;
    *rows = min(max(p.gidx[g], 0), p.M);
  }
}

__device__ __forceinline__ v4f stream_add_slices(const float* at, int64_t stride, int slices) {
  v4f sum = {0.f, 0.f, 0.f, 0.f};
  for (int s0 = 0; s0 < slices; s0 += kReduceBatch) {
    v4f part[kReduceBatch];
#pragma unroll
    for (int i = 0; i < kReduceBatch; ++i)
      if (s0 + i < slices) part[i] = *reinterpret_cast<const v4f_el*>(at + (s0 + i) * stride);
#pragma unroll
    for (int i = 0; i < kReduceBatch; ++i)
      if (s0 + i < slices) sum += part[i];
  }
  return sum;
}

// grid (blocks, experts): silu(gate) * up of the summed row and its 1 x 128 quantiser, 16 lanes per output group.  The sums pass
// through bf16 as the plain GEMM would have stored them, so codes and scales have the bits of the separate steps.
template <int EPI>
__global__ void __launch_bounds__(256) fp8_stream_reduce_act_kernel(const Args p) {
  int row0, rows;
  stream_expert_rows(p, blockIdx.y, &row0, &rows);
  const int lane = threadIdx.x & 63, sub = lane & 15;
  const int gpr = p.act_cols / kScaleBlock;
  const int total = rows * gpr;  // host: partial sums of rows x N floats fit the workspace
  for (int base = (static_cast<int>(blockIdx.x) * 4 + static_cast<int>(threadIdx.x >> 6)) * 4; base < total; base += static_cast<int>(gridDim.x) * 16) {
    const int item = min(base + (lane >> 4), total - 1);
    const int row = item / gpr, kg = item - row * gpr;
    const float* at = p.ws + static_cast<int64_t>(row0 + row) * p.N + kg * kScaleBlock + sub * 8;
    float v[8];
    float amax = 0.f;
#pragma unroll
    for (int half = 0; half < 2; ++half) {
      const v4f gate4 = stream_add_slices(at + 4 * half, p.c_gs, p.splitk);
      const v4f up4 = stream_add_slices(at + p.act_cols + 4 * half, p.c_gs, p.splitk);
#pragma unroll
      for (int j = 0; j < 4; ++j) {
        const float gate = static_cast<float>(static_cast<__bf16>(gate4[j]));
        const float up = static_cast<float>(static_cast<__bf16>(up4[j]));
        float r;
        if (EPI == kSiluQuantMasked)
          r = static_cast<float>(static_cast<__bf16>(up * static_cast<float>(static_cast<__bf16>(act_silu_f32(gate)))));
        else
          r = static_cast<float>(static_cast<__bf16>(act_silu_f32(gate) * up));
        v[4 * half + j] = r;
        amax = fmaxf(amax, fabsf(r));
      }
    }
#pragma unroll
    for (int off = 8; off >= 1; off >>= 1) amax = fmaxf(amax, __shfl_xor(amax, off, 16));
    const float scale = fmaxf(amax, p.act_eps) / 448.0f;
    const float inv_scale = 1.0f / scale;
    int packed[2];
#pragma unroll
    for (int i = 0; i < 2; ++i) {
      float c4[4];
#pragma unroll
      for (int j = 0; j < 4; ++j) c4[j] = fminf(fmaxf(act_div_by_scale(v[4 * i + j], scale, inv_scale), -448.0f), 448.0f);
      int wd = __builtin_amdgcn_cvt_pk_fp8_f32(c4[0], c4[1], 0, false);
      packed[i] = __builtin_amdgcn_cvt_pk_fp8_f32(c4[2], c4[3], wd, true);
    }
    if (base + (lane >> 4) < total) {
      *reinterpret_cast<v2i*>(static_cast<uint8_t*>(p.c) + static_cast<int64_t>(row0 + row) * p.act_q_stride + kg * kScaleBlock + sub * 8) = v2i{packed[0], packed[1]};
      if (sub == 0) {
        const int64_t s_at = p.row_start != nullptr ? static_cast<int64_t>(row0 + row) * p.act_s_sm
                                                    : static_cast<int64_t>(blockIdx.y) * p.act_s_gs + static_cast<int64_t>(row) * p.act_s_sm;
        p.act_s[s_at + static_cast<int64_t>(kg) * p.act_s_sk] = scale;
      }
    }
  }
}

}  // namespace dlb
