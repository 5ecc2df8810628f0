// FP8 block-scaled GEMM for gfx950 in tiles of 128 x 64, for problems with too few of the larger tiles for the chip
// (fp8_gemm_ring.h): 32x32x64 e4m3 MFMA, tiles streamed HBM -> LDS by the DMA path of the memory pipeline
// (global_load_lds_dwordx4, no VGPR staging), multi-stage LDS ring, one barrier per 128-wide K step, block scales applied with
// one FMA per accumulator element and K step.  Also what both files share: DMA and wait primitives, the pre-passes.
//
// Workgroup = WGM x WGN waves, one wave per SIMD; a wave owns MF x NF fragments of 32 x 32 outputs.
// MFMA operand roles: "A" = 32 rows of the weight tile (n), "B" = 32 rows of the activation tile (m), so a lane's
// 16 accumulator components of a fragment are 4 groups of 4 consecutive n for ONE m (= lane & 31): the activation
// scale is one value per lane and fragment row block, and every lane stores 4 contiguous outputs at a time.
//
// Arithmetic: fp8_gemm_kernel of the reference (dlblas/kernels/fp8_gemm.py:49-60).  Requires K % 128 == 0.
#pragma once

#include <type_traits>

#include "fp8_gemm_common.h"
#include "fp8_gemm_tiled.h"  // xcd_remap

namespace dlb {

// D = A_op * B_op^T, A_op / B_op [32 x 64] e4m3: lane l supplies row (l & 31), 32 K-bytes selected by (l >> 5).
// Lane l receives D[8 * (t / 4) + 4 * (l >> 5) + (t % 4)][l & 31] in component t.
__device__ __forceinline__ v16f mfma_32x32x64_e4m3(v8i a_op, v8i b_op, v16f c) {
  return __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a_op, b_op, c, 0, 0, 0, 0, 0, 0);
}

// XOR pattern of the 16-byte chunk index inside a 128-byte LDS row: distinct within any 8 consecutive rows, and
// rows r and r + 8 that share a pattern differ in row parity, i.e. in the 128-byte half of a 256-byte bank line.
__device__ __forceinline__ int chunk_swizzle(int row) { return (row & 7) ^ ((row >> 3) & 1); }

__device__ __forceinline__ int lds_off32(int row, int chunk) {
  return row * kScaleBlock + ((chunk ^ chunk_swizzle(row)) << 4);
}

// A lane reads four 16-byte chunks of "its" row (lane & 31) of every 32-row fragment: logical chunks 2 h, 2 h + 1
// (K half 0) and 4 + 2 h, 5 + 2 h (K half 1), h = lane >> 5.  Fragments start at multiples of 32 rows, which leaves
// the swizzle untouched, so these four byte offsets are the same for every fragment of every tile.
struct LaneChunks {
  int off[4];
};

__device__ __forceinline__ LaneChunks make_lane_chunks(int l32, int h) {
  LaneChunks lc;
#pragma unroll
  for (int i = 0; i < 4; ++i) lc.off[i] = lds_off32(l32, (i >> 1) * 4 + 2 * h + (i & 1));
  return lc;
}

// 8 VGPRs = the 32 operand bytes of one lane for the fragment whose first row starts `frag_bytes` into the LDS
// ring (wave-uniform) and K half `kk` of the 128-byte step.
__device__ __forceinline__ v8i lds_read_frag32(const uint8_t* ring, int frag_bytes, const LaneChunks& lc, int kk) {
  const v4i lo = *reinterpret_cast<const v4i*>(ring + frag_bytes + lc.off[2 * kk]);
  const v4i hi = *reinterpret_cast<const v4i*>(ring + frag_bytes + lc.off[2 * kk + 1]);
  return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
}

typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef __attribute__((address_space(3))) uint8_t* lds_bytes_t;
typedef const __attribute__((address_space(1))) void* global_ptr_t;

// Cache policy operand of the DMA instruction: kDmaStream sets the non-temporal bit.  It is for bytes that few
// workgroups ask for: a chip-wide stream of 256-row panels from HBM runs at 7.1 TB/s with it and 6.1 TB/s without
// (the lines are not kept in the L2 ahead of others), while operands that an XCD's workgroups share through the L2
// lose by it (dense 4096 x 7168 x 18432: 3 % slower with it on the weights, 15 % on both operands).
constexpr int kDmaKeep = 0, kDmaStream = 2;

// One wave-wide DMA: lane i moves 16 bytes from (base + voff) to lds_dst + 16 i.
template <int POLICY = kDmaKeep>
__device__ __forceinline__ void dma_16(const uint8_t* base, uint32_t voff, uint8_t* lds_dst) {
  __builtin_amdgcn_global_load_lds((global_ptr_t)(base + voff), (lds_ptr_t)lds_dst, 16, 0, POLICY);
}
// lane i moves 4 bytes from (base + voff) to lds_dst + 4 i.
template <class LdsPtr>
__device__ __forceinline__ void dma_4(const uint8_t* base, uint32_t voff, LdsPtr lds_dst) {
  __builtin_amdgcn_global_load_lds((global_ptr_t)(base + voff), (lds_ptr_t)lds_dst, 4, 0, 0);
}

template <int POLICY, class LdsPtr>
__device__ __forceinline__ void buf_dma_16(__amdgpu_buffer_rsrc_t rsrc, uint32_t voff, uint32_t soff, LdsPtr lds_dst) {
  __builtin_amdgcn_raw_ptr_buffer_load_lds(rsrc, (lds_ptr_t)lds_dst, 16, voff, soff, 0, POLICY);
}

__device__ __forceinline__ __amdgpu_buffer_rsrc_t make_rsrc(const uint8_t* base, uint32_t bytes) {
  return __builtin_amdgcn_make_buffer_rsrc(const_cast<uint8_t*>(base), 0, bytes, 0x00020000);
}

template <int N>
__device__ __forceinline__ void wait_vmcnt() {
  // s_waitcnt with only vmcnt constrained: vmcnt = simm16[3:0] | simm16[15:14] << 4, expcnt [6:4], lgkmcnt [11:8]
  __builtin_amdgcn_s_waitcnt((N & 0xF) | (((N >> 4) & 0x3) << 14) | (0x7 << 4) | (0xF << 8));
}

// Workgroup barrier that orders LDS traffic only: every wave's LDS reads have returned (lgkmcnt) before it
// arrives.  Unlike __syncthreads() it does not drain the vector-memory counter, so DMA groups that were issued
// for later stages stay in flight across it; the caller waits for the group it needs with wait_vmcnt first.
__device__ __forceinline__ void lds_barrier() { asm volatile("s_waitcnt lgkmcnt(0)\n\ts_barrier" ::: "memory"); }

// Four floats to / from memory that another workgroup of the same launch reads / wrote: device-scope accesses
// (write-through, and read past the caches that are not coherent between the XCDs), 8 bytes each, relaxed.
__device__ __forceinline__ void coherent_store16(float* dst, v4f v) {
  typedef float v2f __attribute__((ext_vector_type(2)));
  uint64_t* d = reinterpret_cast<uint64_t*>(dst);
  __hip_atomic_store(d, __builtin_bit_cast(uint64_t, v2f{v.x, v.y}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
  __hip_atomic_store(d + 1, __builtin_bit_cast(uint64_t, v2f{v.z, v.w}), __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
}
__device__ __forceinline__ v4f coherent_load16(const float* src) {
  typedef float v2f __attribute__((ext_vector_type(2)));
  const uint64_t* s = reinterpret_cast<const uint64_t*>(src);
  const v2f lo = __builtin_bit_cast(v2f, __hip_atomic_load(s, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  const v2f hi = __builtin_bit_cast(v2f, __hip_atomic_load(s + 1, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT));
  return v4f{lo.x, lo.y, hi.x, hi.y};
}

// f(0), f(1), ... with compile-time indices
template <class F, int... I>
__device__ __forceinline__ void each_index(F&& f, std::integer_sequence<int, I...>) {
  (f(std::integral_constant<int, I>{}), ...);
}

// One wave per SIMD, 512 registers: every fragment of the NEXT K step is read into a second register set while the current step
// computes, so no MFMA of a step waits for LDS.
// SCTAB_: true = the activation scales of a tile's rows for ALL K blocks of the workgroup's K range (at most
// SCTAB_KB) are fetched once per tile into a table behind the ring, lanes along K: a row-major a_s then costs one
// cache-line request per row and tile instead of one per row and K step, and needs no re-layout pass in front.
template <int WGM_, int WGN_, int MF_, int NF_, int STAGES_, bool SCTAB_ = false, int SCTAB_KB_ = 32>
struct PipeCfg {
  static constexpr int WGM = WGM_, WGN = WGN_, MF = MF_, NF = NF_, STAGES = STAGES_;
  static constexpr bool SCTAB = SCTAB_;
  static constexpr int WAVES = WGM * WGN;
  static constexpr int NT = WAVES * 64;
  static constexpr int BM = WGM * MF * 32;
  static constexpr int BN = WGN * NF * 32;
  static constexpr int A_INST = BM / 8 / WAVES;  // 16-byte DMA instructions per wave and stage for the A tile
  static constexpr int B_INST = BN / 8 / WAVES;
  static constexpr int S_INST = SCTAB ? 0 : (BM + NT - 1) / NT;  // 4-byte DMA instructions per wave for the a_s slice
  static constexpr int A_BYTES = BM * kScaleBlock;
  static constexpr int B_BYTES = BN * kScaleBlock;
  static constexpr int S_BYTES = S_INST * NT * 4;  // activation scales of the tile rows for one K block
  static constexpr int W_BYTES = NT * 4;           // weight scale of each wave's n block, one copy per lane
  static constexpr int STAGE_BYTES = A_BYTES + B_BYTES + S_BYTES + W_BYTES;
  static constexpr int SCTAB_KB = SCTAB_KB_;       // K blocks per workgroup the table holds
  static constexpr int SCTAB_OFF = STAGES * STAGE_BYTES;
  static constexpr int SCTAB_BYTES = SCTAB ? BM * (SCTAB_KB + 1) * 4 : 0;  // rows of an odd pitch (bank spread), at most SCTAB_KB + 1 floats
  static constexpr int LDS_BYTES = STAGES * STAGE_BYTES + SCTAB_BYTES;
  static constexpr int LOADS_PER_STAGE = A_INST + B_INST + S_INST + 1;  // vmcnt units per wave and stage
  static_assert(BM % (8 * WAVES) == 0 && BN % (8 * WAVES) == 0, "tile rows must divide over the DMA instructions");
  static_assert(128 % (NF * 32) == 0, "a wave's columns share one weight scale");
  static_assert(MF * NF <= 4, "both fragment sets fit the registers");
  static_assert(LOADS_PER_STAGE * (STAGES - 1) < 64, "vmcnt is a 6-bit counter");
};

// Re-lays activation scales from [groups][rows][kblocks] (any strides) to [groups][kblocks][rows_pad], rows
// contiguous, so that the GEMM's per-K-step fetch of one scale per tile row is a handful of full cache lines
// instead of one line per row.  32 x 32 tiles through LDS keep both sides coalesced.  (The reference does the same
// re-layout before its grouped GEMMs, dlblas/kernels/quant_dequant.py:42-83.)
// rows_map (or NULL): row r of the re-laid copy is row rows_map[r] of src.  (bx, by, g): the block's 32 x 32 tile and group.
__device__ __forceinline__ void scale_transpose_block(const float* src, float* dst, int rows, int kblocks, int rows_pad,
                                                      int64_t s_g, int64_t s_m, int64_t s_k, const int32_t* rows_map, int bx,
                                                      int by, int g) {
  __shared__ float tile[32][33];
  const int r0 = bx * 32, k0 = by * 32;
  const int tx = threadIdx.x & 31, ty = threadIdx.x >> 5;  // 32 x 8
  const float* in = src + static_cast<int64_t>(g) * s_g;
  float* out = dst + static_cast<int64_t>(g) * kblocks * rows_pad;
#pragma unroll
  for (int i = 0; i < 32; i += 8) {
    const int r = r0 + ty + i, k = k0 + tx;
    const bool live = r < rows && k < kblocks;
    const int64_t sr = (live && rows_map != nullptr) ? max(rows_map[r], 0) : r;
    tile[ty + i][tx] = live ? in[sr * s_m + static_cast<int64_t>(k) * s_k] : 0.f;
  }
  __syncthreads();
#pragma unroll
  for (int i = 0; i < 32; i += 8) {
    const int k = k0 + ty + i, r = r0 + tx;
    if (k < kblocks && r < rows_pad) out[static_cast<int64_t>(k) * rows_pad + r] = tile[tx][ty + i];
  }
}

__global__ void __launch_bounds__(256) fp8_scale_transpose_kernel(const float* src, float* dst, int rows, int kblocks,
                                                                  int rows_pad, int64_t s_g, int64_t s_m, int64_t s_k,
                                                                  const int32_t* rows_map) {
  scale_transpose_block(src, dst, rows, kblocks, rows_pad, s_g, s_m, s_k, rows_map, blockIdx.x, blockIdx.y, blockIdx.z);
}

constexpr int kTileListHeader = 3;  // tile counts in front of the three tile lists of an expert-contiguous launch

// Work of one workgroup: tiles vb_first, vb_first + gridDim.x, ... of tiles_m x tiles_n tiles of BM x BN.
template <class Cfg, int MODE>
__device__ __forceinline__ void pipelined_body(const Args& p, uint8_t* smem, int vb_first, int tiles_m, int tiles_n) {
  constexpr int BM = Cfg::BM, BN = Cfg::BN, MF = Cfg::MF, NF = Cfg::NF, WAVES = Cfg::WAVES, STAGES = Cfg::STAGES;
  // Grouped modes: an expert's weight tile is read by the one to three row tiles of that expert, not by a column of
  // the grid: streamed (2 - 7 % faster from 128 to 768 rows per expert at 32 x 4096 x 7168).
  constexpr int kWeightPolicy = MODE == kDense ? kDmaKeep : kDmaStream;

  const int tid = threadIdx.x;
  const int lane = tid & 63;
  const int wave = __builtin_amdgcn_readfirstlane(tid >> 6);
  const int l32 = lane & 31;
  const int h = lane >> 5;
  const int wm0 = (wave / Cfg::WGN) * (MF * 32);
  const int wn0 = (wave % Cfg::WGN) * (NF * 32);
  const LaneChunks lc = make_lane_chunks(l32, h);

  const int tiles = tiles_m * tiles_n;
  int walk_g = 0;
  int walk_base = 0;
  // Unit id of a dense launch: the tile, in patches of group_m row tiles, and the slice of K.  The K range is cut into
  // p.splitk slices of p.kb_per_split blocks; slices of one tile are far apart in the order.
  const int units = MODE == kDense ? tiles * p.splitk : tiles;
  auto locate = [&](int v, int& tile, int& slice, int& tm, int& tn) __attribute__((always_inline)) {
    const int id = xcd_remap(v, units);
    slice = MODE == kDense ? id / tiles : 0;
    tile = id - slice * tiles;
    const int width = p.group_m * tiles_n;
    const int grp = tile / width;
    const int first_m = grp * p.group_m;
    const int gsz = min(tiles_m - first_m, p.group_m);
    const int in_grp = tile - grp * width;
    tm = first_m + in_grp % gsz;
    tn = in_grp / gsz;
  };
  for (int vb = vb_first;; vb += gridDim.x) {
    int g = 0, mt = 0, nt, m_end, split = 0, tile_lin = 0;
    if (MODE == kMasked) {
      // The tile count is only known on the device, so the grid is persistent; the hardware deals consecutive
      // workgroups to the 8 XCDs in turn.  Of every 32 consecutive tiles each XCD takes 4 consecutive ones: the row
      // tiles of an expert, which are adjacent in the order and read the same weight tile, meet in one L2, and the
      // last, partial round still spreads over all XCDs (the grid is a multiple of 32).
      const int grid = static_cast<int>(gridDim.x);
      const int w = vb % grid;
      const int tile_id = vb - w + (w / 32) * 32 + (w % 8) * 4 + (w / 8) % 4;
      int mtiles = 0;
      while (walk_g < p.G) {
        const int valid = min(max(p.gidx[walk_g], 0), p.M);
        mtiles = (valid + BM - 1) / BM;
        const int cnt = mtiles * tiles_n;
        if (tile_id < walk_base + cnt) break;
        walk_base += cnt;
        ++walk_g;
      }
      if (walk_g >= p.G) break;
      g = walk_g;
      const int local = tile_id - walk_base;
      mt = local % mtiles;
      nt = local / mtiles;
      m_end = min(max(p.gidx[g], 0), p.M);
    } else {
      if (vb >= units) break;
      locate(vb, tile_lin, split, mt, nt);
      m_end = p.M;
      if (MODE == kContiguous) {
        g = p.gidx[mt * BM];
        if (g < 0 || g >= p.G) continue;
      }
    }
    g = __builtin_amdgcn_readfirstlane(g);
    const int m0 = __builtin_amdgcn_readfirstlane(mt * BM);
    const int n0 = __builtin_amdgcn_readfirstlane(nt * BN);

    const int64_t esz = p.out_f32 ? 4 : 2;
    const bool sliced = MODE == kDense && p.splitk > 1;
    const int kb_first = sliced ? split * p.kb_per_split : 0;  // the host leaves no slice empty
    const int nk = sliced ? min(p.kblocks, kb_first + p.kb_per_split) - kb_first : p.kblocks;  // K blocks of this unit
    const uint8_t* a_tile = p.a + static_cast<int64_t>(m0) * p.K + static_cast<int64_t>(kb_first) * kScaleBlock;
    const float* as_tile = p.a_s + static_cast<int64_t>(m0) * p.as_sm + static_cast<int64_t>(kb_first) * p.as_sk;
    char* c_base = static_cast<char*>(p.c);
    if (MODE == kMasked) {
      a_tile += static_cast<int64_t>(g) * p.a_gs;
      as_tile += static_cast<int64_t>(g) * p.as_gs;
      c_base += static_cast<int64_t>(g) * p.c_gs * esz;
    }
    const uint8_t* b_tile = p.b + static_cast<int64_t>(g) * p.b_gs + static_cast<int64_t>(n0) * p.K +
                            static_cast<int64_t>(kb_first) * kScaleBlock;
    // the wave's weight scale, fetched by every lane
    const float* bs_g = p.b_s + static_cast<int64_t>(g) * p.bs_gs + kb_first;
    const uint32_t bs_off = static_cast<uint32_t>(min((n0 + wn0) / kScaleBlock, p.nblocks - 1)) * static_cast<uint32_t>(p.kblocks) * 4u;

    // DMA addressing.  Instruction j of this wave fills LDS rows 8 (j WAVES + wave) .. + 7; lane i fills physical
    // chunk (i & 7) of row (i >> 3), which holds logical chunk (i & 7) ^ swizzle(row).  WAVES is even, so the
    // swizzle does not depend on j and one per-lane chunk offset serves every instruction; the row part is
    // recomputed per instruction (two VALU ops) instead of being kept in registers.  Rows past the valid range
    // re-read the last valid row.
    static_assert(WAVES % 2 == 0, "chunk swizzle must not depend on the DMA instruction index");
    const int a_last = m_end - 1 - m0;
    const int b_last = p.N - 1 - n0;
    const int dma_row = 8 * wave + (lane >> 3);
    const uint32_t dma_chunk = static_cast<uint32_t>(((lane & 7) ^ chunk_swizzle(dma_row)) * 16);
    const uint32_t uK = static_cast<uint32_t>(p.K);

    // Per-lane source offsets of every DMA instruction of a stage, computed once per tile: the K loop then issues
    // its DMA group without any vector ALU work (32-bit multiplies are quarter rate and, issued right behind the
    // barrier by every wave at once, kept the matrix pipe waiting).
    uint32_t a_off[Cfg::A_INST], b_off[Cfg::B_INST], s_off[Cfg::S_INST > 0 ? Cfg::S_INST : 1];
#pragma unroll
    for (int j = 0; j < Cfg::A_INST; ++j) {
      const int r = min(dma_row + 8 * j * WAVES, a_last);
      a_off[j] = static_cast<uint32_t>(r) * uK + dma_chunk;
    }
#pragma unroll
    for (int j = 0; j < Cfg::B_INST; ++j)
      b_off[j] = static_cast<uint32_t>(min(dma_row + 8 * j * WAVES, b_last)) * uK + dma_chunk;
#pragma unroll
    for (int j = 0; j < Cfg::S_INST; ++j)
      s_off[j] = static_cast<uint32_t>(min((j * WAVES + wave) * 64 + lane, a_last)) * static_cast<uint32_t>(p.as_sm) * 4u;

    auto issue_stage = [&](int kb, int stage) {
      uint8_t* sbase = smem + stage * Cfg::STAGE_BYTES;
      const uint8_t* ag = a_tile + static_cast<int64_t>(kb) * kScaleBlock;
      const uint8_t* bg = b_tile + static_cast<int64_t>(kb) * kScaleBlock;
      const uint8_t* sg = reinterpret_cast<const uint8_t*>(as_tile + static_cast<int64_t>(kb) * p.as_sk);
      // the empty asm keeps each offset a 32-bit register here, so that the load uses the scalar-base + 32-bit
      // vector-offset form instead of a 64-bit address built outside the loop (two registers per instruction)
#pragma unroll
      for (int j = 0; j < Cfg::A_INST; ++j) {
        uint32_t o = a_off[j];
        asm volatile("" : "+v"(o));
        dma_16(ag, o, sbase + (j * WAVES + wave) * 1024);
      }
#pragma unroll
      for (int j = 0; j < Cfg::B_INST; ++j) {
        uint32_t o = b_off[j];
        asm volatile("" : "+v"(o));
        dma_16<kWeightPolicy>(bg, o, sbase + Cfg::A_BYTES + (j * WAVES + wave) * 1024);
      }
#pragma unroll
      for (int j = 0; j < Cfg::S_INST; ++j) {
        uint32_t o = s_off[j];
        asm volatile("" : "+v"(o));
        dma_4(sg, o, sbase + Cfg::A_BYTES + Cfg::B_BYTES + (j * WAVES + wave) * 256);
      }
      // weight scale of the wave's columns at this K block
      dma_4(reinterpret_cast<const uint8_t*>(bs_g + kb), bs_off,
            sbase + Cfg::A_BYTES + Cfg::B_BYTES + Cfg::S_BYTES + wave * 256);
    };

    v16f acc[MF][NF];
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int ni = 0; ni < NF; ++ni)
#pragma unroll
        for (int t = 0; t < 16; ++t) acc[mi][ni][t] = 0.f;

    // ---- K loop ---------------------------------------------------------------------------------------------
    constexpr int T = MF * NF;
    constexpr int kFragBytes = 32 * kScaleBlock;
    constexpr int kScaleOff = Cfg::A_BYTES + Cfg::B_BYTES;
    constexpr int kWScaleOff = kScaleOff + Cfg::S_BYTES;

    // scale table [BM][p.sct_pitch]: entry (r, j) = a_s of tile row r at the workgroup's j-th K block.  One DMA
    // instruction moves 64 consecutive entries, i.e. whole runs of a row's scales; issued ahead of the first stages,
    // so the wait for stage 0 covers them.  The pitch is odd: the 32 rows a wave reads at one K block then lie in 32
    // different banks (with a power-of-two pitch of 32 floats they shared two banks, and every such read held the
    // LDS for 16 turns while the other waves' fragment reads waited: 256 x 7168 x 4096 27.2 -> 24 us).
    auto issue_table = [&]() __attribute__((always_inline)) {
      const int pitch = p.sct_pitch;
      const float inv_pitch = 1.0f / static_cast<float>(pitch);
      const int n_inst = (BM * pitch + 63) >> 6;
      for (int i = wave; i < n_inst; i += WAVES) {
        const int e = i * 64 + lane;
        const int row = static_cast<int>((static_cast<float>(e) + 0.5f) * inv_pitch);  // e / pitch, exact for e < 2^20
        const uint32_t r = static_cast<uint32_t>(min(row, a_last));
        const uint32_t j = static_cast<uint32_t>(min(e - row * pitch, nk - 1));
        dma_4(reinterpret_cast<const uint8_t*>(as_tile),
              (r * static_cast<uint32_t>(p.as_sm) + j * static_cast<uint32_t>(p.as_sk)) * 4u, smem + Cfg::SCTAB_OFF + i * 256);
      }
    };
    int stage = 0;
    __syncthreads();  // the previous tile's readers are done with the ring
    if constexpr (Cfg::SCTAB) issue_table();
#pragma unroll
    for (int s = 0; s < STAGES; ++s)
      if (s < nk) issue_stage(s, s);
    // all but the first stage's group may still be on their way
    if (nk >= STAGES)
      wait_vmcnt<(STAGES - 1) * Cfg::LOADS_PER_STAGE>();
    else
      wait_vmcnt<0>();
    lds_barrier();

    // first table entry of this lane's rows (scale-table kernels)
    int tab_row[MF];
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) tab_row[mi] = Cfg::SCTAB ? (wm0 + mi * 32 + l32) * p.sct_pitch : 0;

    v8i xr[2][MF][2];
    v8i wr[2][NF][2];
    float scb[2][MF];
    float sc_last = 0.f;
    v16f part[2];
#pragma unroll
    for (int u = 0; u < 16; ++u) part[0][u] = part[1][u] = 0.f;
    const int x0 = wm0 * kScaleBlock;
    const int w0 = (Cfg::BM + wn0) * kScaleBlock;
    auto load_scales = [&](int base, int kbl, float (&dst)[MF]) {
      const float sb = *reinterpret_cast<const float*>(smem + base + kWScaleOff + wave * 256);
      if constexpr (Cfg::SCTAB) {
        const float* tab = reinterpret_cast<const float*>(smem + Cfg::SCTAB_OFF);
#pragma unroll
        for (int mi = 0; mi < MF; ++mi) dst[mi] = tab[tab_row[mi] + kbl] * sb;
      } else {
        const float* sS = reinterpret_cast<const float*>(smem + base + kScaleOff);
#pragma unroll
        for (int mi = 0; mi < MF; ++mi) dst[mi] = sS[wm0 + mi * 32 + l32] * sb;
      }
    };
    // half-fragment q of a stage: q < 2 MF -> activation fragment q / 2, K half q % 2; else weight fragment
    constexpr int kHalves = 2 * (MF + NF);
    constexpr int kPerTile = (kHalves + (MF * NF) - 2) / (MF * NF - 1);  // spread over the first T - 1 tiles
    load_scales(0, 0, scb[0]);
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      xr[0][mi][0] = lds_read_frag32(smem, x0 + mi * kFragBytes, lc, 0);
      xr[0][mi][1] = lds_read_frag32(smem, x0 + mi * kFragBytes, lc, 1);
    }
#pragma unroll
    for (int ni = 0; ni < NF; ++ni) {
      wr[0][ni][0] = lds_read_frag32(smem, w0 + ni * kFragBytes, lc, 0);
      wr[0][ni][1] = lds_read_frag32(smem, w0 + ni * kFragBytes, lc, 1);
    }

    // Every step is the same code: a step always prefetches "the next stage" into registers (garbage after the
    // last one, never used); whether it hands its stage to the DMA and how many groups it leaves in flight at its
    // barrier are wave-uniform branches on the step's distance from the end of K.
    auto k_step = [&](auto buf_tag, int kb, int stage) __attribute__((always_inline)) {
      constexpr int B = decltype(buf_tag)::value;
      const int next_stage = stage + 1 == STAGES ? 0 : stage + 1;
      const int nxt_base = next_stage * Cfg::STAGE_BYTES;
      // every wave holds this stage's fragments in registers and has its share of the next stage in LDS
      // the group of step kb + 1 has landed: behind it at most STAGES - 2 younger groups are out, fewer at the tile's end
      if (kb + STAGES > nk)
        wait_vmcnt<0>();
      else
        wait_vmcnt<(STAGES - 2) * Cfg::LOADS_PER_STAGE>();
      lds_barrier();
      if (kb + STAGES < nk) issue_stage(kb + STAGES, stage);
#pragma unroll
      for (int t = 0; t < T; ++t) {
        const int mi = t / NF, ni = t % NF;
        __builtin_amdgcn_sched_barrier(0);
        v16f z;
#pragma unroll
        for (int u = 0; u < 16; ++u) z[u] = 0.f;
        z = mfma_32x32x64_e4m3(wr[B][ni][0], xr[B][mi][0], z);
        part[t & 1] = mfma_32x32x64_e4m3(wr[B][ni][1], xr[B][mi][1], z);
        __builtin_amdgcn_sched_barrier(0);
        if (t == 0) load_scales(nxt_base, min(kb + 1, nk - 1), scb[B ^ 1]);
#pragma unroll
        for (int q = t * kPerTile; q < (t + 1) * kPerTile && q < kHalves; ++q) {
          if (q < 2 * MF)
            xr[B ^ 1][q / 2][q % 2] = lds_read_frag32(smem, nxt_base + x0 + (q / 2) * kFragBytes, lc, q % 2);
          else
            wr[B ^ 1][(q - 2 * MF) / 2][q % 2] =
                lds_read_frag32(smem, nxt_base + w0 + ((q - 2 * MF) / 2) * kFragBytes, lc, q % 2);
        }
        __builtin_amdgcn_sched_barrier(0);
        if (t == 0)
          acc[MF - 1][NF - 1] += part[(T - 1) & 1] * sc_last;  // last tile of the previous K step
        else
          acc[(t - 1) / NF][(t - 1) % NF] += part[(t - 1) & 1] * scb[B][(t - 1) / NF];
      }
      sc_last = scb[B][MF - 1];
    };
    typedef std::integral_constant<int, 0> B0;
    typedef std::integral_constant<int, 1> B1;
    int kb = 0;
    for (; kb + 1 < nk; kb += 2) {
      k_step(B0{}, kb, stage);
      stage = stage + 1 == STAGES ? 0 : stage + 1;
      k_step(B1{}, kb + 1, stage);
      stage = stage + 1 == STAGES ? 0 : stage + 1;
    }
    if (kb < nk) k_step(B0{}, kb, stage);
    acc[MF - 1][NF - 1] += part[(T - 1) & 1] * sc_last;

    // epilogue: lane holds c[m0 + wm0 + 32 mi + (lane & 31)][n0 + wn0 + 32 ni + 8 u + 4 (lane >> 5) + 0..3], u = 0..3
    const int el = lane, el32 = lane & 31, eh = lane >> 5;
    if (sliced && p.fused_reduce) {
      // Split-K in one launch.  The workgroups of a tile (one per K slice) park their fp32 sums in the workspace,
      // count themselves in on the tile's arrival counter, wait - for a bounded time - until all slices are in, and
      // then each adds up its share of the tile: the slices in index order (the same order, and so the same bits, as
      // fp8_splitk_reduce_kernel), cast, store.  Nobody depends on that wait for correctness: a workgroup that gives
      // up sets its bit in the tile's word of abandoned shares and looks at the counter once more (all in after all:
      // it adds its share anyway); the workgroup whose arrival completed the tile reads that word after its own share
      // and adds the shares named there.  A share that both of them add is stored twice with the same bits.  The last
      // workgroup to leave the tile zeroes its three counters: the workspace head is all zero when the launch ends.
      // Partial sums are written in accumulator order: unit ((wave MF + mi) NF + ni) 4 + u holds, for lane l, the four
      // floats c[32 mi + (l & 31)][32 ni + 8 u + 4 (l >> 5) + 0..3] of that wave's tile.
      constexpr int kTileFloats = BM * BN;
      constexpr int kUnits = kTileFloats / 4;
      const int S = p.splitk;
      float* tbase = p.ws + static_cast<int64_t>(tile_lin) * S * kTileFloats;
      float* mine = tbase + static_cast<int64_t>(split) * kTileFloats;
#pragma unroll
      for (int mi = 0; mi < MF; ++mi)
#pragma unroll
        for (int ni = 0; ni < NF; ++ni)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const v4f v = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
            coherent_store16(mine + ((((wave * MF + mi) * NF + ni) * 4 + u) * 64 + lane) * 4, v);
          }
      // The stores above are write-through, device-scope stores: once the memory counter has drained they are where
      // every XCD reads them.  (A release fence here would also write back the whole L2 of this XCD, once per
      // workgroup: measured at 4 - 11 us per launch.)
      asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      __syncthreads();  // ... those of every wave; the ring is idle from here on
      uint32_t* ctr = p.ctr + static_cast<int64_t>(tile_lin) * 4;
      volatile uint32_t* flag = reinterpret_cast<volatile uint32_t*>(smem);
      const uint32_t uS = static_cast<uint32_t>(S);
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
          __hip_atomic_fetch_or(ctr + 1, 1u << split, __ATOMIC_SEQ_CST, __HIP_MEMORY_SCOPE_AGENT);
          all_in = __hip_atomic_load(ctr, __ATOMIC_SEQ_CST, __HIP_MEMORY_SCOPE_AGENT) >= uS;
        }
        flag[0] = all_in ? 1u << split : 0u;
        flag[1] = last ? 1u : 0u;
      }
      __syncthreads();
      const bool last = flag[1] != 0;
      const int64_t esz_c = p.out_f32 ? 4 : 2;
      auto add_unit = [&](int u, const v4f& sum) {
        const int ul = u & 63, uu = (u >> 6) & 3, f = u >> 8;  // f = (wave MF + mi) NF + ni
        const int fni = f % NF, fmi = (f / NF) % MF, fw = f / (NF * MF);
        const int m = m0 + (fw / Cfg::WGN) * (MF * 32) + fmi * 32 + (ul & 31);
        const int n = n0 + (fw % Cfg::WGN) * (NF * 32) + fni * 32 + uu * 8 + (ul >> 5) * 4;
        if (m >= m_end) return;
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
        for (int j = 0; j < S; ++j) {
          if (!((todo >> j) & 1u)) continue;
          const int u0 = static_cast<int>(static_cast<int64_t>(j) * kUnits / S);
          const int u1 = static_cast<int>(static_cast<int64_t>(j + 1) * kUnits / S);
          // two units per thread and pass, the loads of up to eight slices of both in flight before the first sum
          for (int ua = u0 + tid; ua < u1; ua += 2 * Cfg::NT) {
            const int ub = ua + Cfg::NT;
            const bool has_b = ub < u1;
            v4f sum_a = {0.f, 0.f, 0.f, 0.f}, sum_b = {0.f, 0.f, 0.f, 0.f};
            for (int sb = 0; sb < S; sb += 8) {
              v4f pa[8], pb[8];
#pragma unroll
              for (int i = 0; i < 8; ++i) {
                pa[i] = pb[i] = v4f{0.f, 0.f, 0.f, 0.f};
                if (sb + i < S) {
                  pa[i] = coherent_load16(tbase + static_cast<int64_t>(sb + i) * kTileFloats + ua * 4);
                  if (has_b) pb[i] = coherent_load16(tbase + static_cast<int64_t>(sb + i) * kTileFloats + ub * 4);
                }
              }
#pragma unroll
              for (int i = 0; i < 8; ++i)
                if (sb + i < S) sum_a += pa[i], sum_b += pb[i];
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
      continue;
    }
    // Results leave through LDS: stored straight from the accumulator layout every instruction would touch 32 rows with
    // 16 or 32 bytes each, partial sectors that the L2 has to merge.  Each wave parks rows of its tile in its own slice
    // of the (now idle) ring, rotated by their index to spread the banks, and reads them back row-wise: a store
    // instruction then writes whole rows, 16 bytes per lane, at whatever alignment N leaves the rows.
    // (us per call: 3779 x 6111 x 1024 bf16, rows at odd addresses that used to leave 2 bytes a store, 95 -> 42; 2000 x 5001 x
    // 4096 fp32 79 -> 53; 3875 x 11520 x 640 fp32, aligned rows, 75 -> 71.)
    const bool cols_inside = n0 + wn0 + NF * 32 <= p.N;  // no column of the wave's tile lies past N: stores without a tail
    auto store_rows_f32 = [&](float* c_tile) __attribute__((always_inline)) {
      // 32 rows of the wave's tile at a time
      constexpr int kRowBytes = NF * 32 * 4;
      constexpr int kCpr = kRowBytes / 16;   // 16-byte chunks per row
      constexpr int kRpi = 64 / kCpr;        // rows per store instruction
      static_assert(32 * kRowBytes * WAVES <= Cfg::LDS_BYTES, "the staging slices fit in the ring");
      uint8_t* st = smem + wave * (32 * kRowBytes);
      const int r_in = el / kCpr, ch = el % kCpr;
      const int n_left = p.N - (n0 + wn0 + ch * 4);
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
#pragma unroll
        for (int ni = 0; ni < NF; ++ni)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const v4f v = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
            *reinterpret_cast<v4f*>(st + el32 * kRowBytes + (ni * 8 + 2 * u + eh + el32) % kCpr * 16) = v;
          }
        // a wave reads only what it wrote: no barrier, the LDS counter orders the two
        auto store_rows = [&](auto inside) __attribute__((always_inline)) {
#pragma unroll 4
          for (int r0 = 0; r0 < 32; r0 += kRpi) {
            const int row = r0 + r_in;
            if (el >= kRpi * kCpr || row >= 32) continue;
            const v4f v = *reinterpret_cast<const v4f*>(st + row * kRowBytes + (ch + row) % kCpr * 16);
            if (m0 + wm0 + mi * 32 + row < m_end) store_row4<true>(c_tile + static_cast<int64_t>(mi * 32 + row) * p.N, ch * 4, v, inside ? 4 : n_left);
          }
        };
        if (cols_inside)
          store_rows(std::true_type{});
        else
          store_rows(std::false_type{});
      }
    };
    if (sliced) {
      // first pass of split-K: the slice's sums go to the workspace as an fp32 [M][N] matrix of their own;
      // fp8_splitk_reduce_kernel, launched behind this kernel on the same stream, adds the slices in index order
      __syncthreads();  // every wave is done reading the ring
      store_rows_f32(p.ws + static_cast<int64_t>(split) * p.M * p.N + static_cast<int64_t>(m0 + wm0) * p.N + n0 + wn0);
      continue;
    }
    if (p.c_lds && p.out_f32) {
      __syncthreads();
      store_rows_f32(reinterpret_cast<float*>(c_base) + static_cast<int64_t>(m0 + wm0) * p.N + n0 + wn0);
      continue;
    }
    if (p.c_lds) {
      constexpr int kRowBytes = NF * 32 * 2;
      constexpr int kCpr = kRowBytes / 16;   // 16-byte chunks per row
      constexpr int kRpi = 64 / kCpr;        // rows per store instruction
      static_assert(MF * 32 * kRowBytes * WAVES <= Cfg::LDS_BYTES, "the staging slices fit in the ring");
      __syncthreads();
      uint8_t* st = smem + wave * (MF * 32 * kRowBytes);
#pragma unroll
      for (int mi = 0; mi < MF; ++mi) {
        const int row = mi * 32 + el32;
#pragma unroll
        for (int ni = 0; ni < NF; ++ni)
#pragma unroll
          for (int u = 0; u < 4; ++u) {
            const v4f v = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
            const int chunk = (ni * 4 + u + row) % kCpr;
            *reinterpret_cast<v4bf*>(st + row * kRowBytes + chunk * 16 + eh * 8) = __builtin_convertvector(v, v4bf);
          }
      }
      const int r_in = el / kCpr, ch = el % kCpr;
      const int n_left = p.N - (n0 + wn0 + ch * 8);
      __bf16* c_tile = reinterpret_cast<__bf16*>(c_base) + static_cast<int64_t>(m0 + wm0) * p.N + n0 + wn0;
      auto store_rows = [&](auto inside) __attribute__((always_inline)) {
#pragma unroll 4
        for (int r0 = 0; r0 < MF * 32; r0 += kRpi) {
          const int row = r0 + r_in;
          if (el >= kRpi * kCpr || row >= MF * 32) continue;
          const v4i v = *reinterpret_cast<const v4i*>(st + row * kRowBytes + ((ch + row) % kCpr) * 16);
          if (m0 + wm0 + row < m_end && (inside || n_left > 0)) store_row8_bf16(c_tile + static_cast<int64_t>(row) * p.N + ch * 8, v, inside ? 8 : n_left);
        }
      };
      if (cols_inside)
        store_rows(std::true_type{});
      else
        store_rows(std::false_type{});
      continue;
    }
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      const int m = m0 + wm0 + mi * 32 + el32;
      if (m >= m_end) continue;
      char* c_row = c_base + static_cast<int64_t>(m) * p.N * esz;
#pragma unroll
      for (int ni = 0; ni < NF; ++ni) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const int n = n0 + wn0 + ni * 32 + u * 8 + eh * 4;
          const v4f v = {acc[mi][ni][4 * u], acc[mi][ni][4 * u + 1], acc[mi][ni][4 * u + 2], acc[mi][ni][4 * u + 3]};
          if (p.out_f32)
            store_row4<true>(c_row, n, v, p.N - n);
          else
            store_row4<false>(c_row, n, v, p.N - n);
        }
      }
    }
  }
}

template <class Cfg, int MODE>
__global__ void __launch_bounds__(Cfg::NT) fp8_gemm_pipelined_kernel(const Args p) {
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  pipelined_body<Cfg, MODE>(p, smem, blockIdx.x, p.tiles_m, p.tiles_n);
}

// Expert-contiguous rows: a one-block pre-pass turns m_indices into three tile lists.  A run of R adjacent 128-row
// blocks of one expert becomes R / 2 tiles of 256 rows when R is even, one tile of 128 rows when R = 1, and
// (R - 3) / 2 tiles of 256 rows followed by two tiles of 192 rows when R is odd: most weight tiles are then fetched
// once per expert instead of once per 128 rows, and the two 192-row tiles of an odd run, which are adjacent in their
// list, run side by side on one XCD at the same pace, so that the second finds the weight tile in the L2 (a 256-row
// and a 128-row tile drift apart and stream it twice).  Blocks whose first index is negative (or not an expert)
// appear in no list.  list layout: [0] = n256, [1] = n192, [2] = n128, then the three lists of `cap` entries each;
// an entry is the tile's first row in units of 64 rows.
constexpr int kTileListMaxBlocks = 4096;  // 512 K rows; more rows fall back to uniform 128-row tiles

__device__ __forceinline__ void contiguous_tile_list_block(const int32_t* m_indices, int M, int G, int32_t* tlist, int cap) {
  __shared__ int eb[kTileListMaxBlocks];   // expert of every 128-row block, -1 = skip
  __shared__ int rs[kTileListMaxBlocks];   // first block of the run of equal experts the block belongs to
  __shared__ int re[kTileListMaxBlocks];   // last block of that run
  __shared__ int chunk_last[256], chunk_first[256];
  __shared__ int n256, n192, n128;
  const int tid = threadIdx.x;
  const int nblk = (M + 127) / 128;
  if (tid == 0) n256 = n192 = n128 = 0;
  for (int b = tid; b < nblk; b += 256) {
    const int e = m_indices[static_cast<int64_t>(b) * 128];
    eb[b] = (e >= 0 && e < G) ? e : -1;
  }
  __syncthreads();
  const int chunk = (nblk + 255) / 256;
  const int b0 = min(nblk, tid * chunk), b1 = min(nblk, b0 + chunk);
  int last = -1;
  for (int b = b0; b < b1; ++b) {
    if (b == 0 || eb[b] != eb[b - 1]) last = b;
    rs[b] = last;
  }
  chunk_last[tid] = last;
  int first = nblk;  // the same from the right: nearest run end at or after the block
  for (int b = b1 - 1; b >= b0; --b) {
    if (b == nblk - 1 || eb[b] != eb[b + 1]) first = b;
    re[b] = first;
  }
  chunk_first[tid] = first;
  __syncthreads();
  // what the chunks before (after) this one carry in: running maximum of chunk_last from the left, running minimum of
  // chunk_first from the right, as two scans over the 256 chunk values in eight steps
  for (int off = 1; off < 256; off <<= 1) {
    const int from_left = tid >= off ? chunk_last[tid - off] : -1;
    const int from_right = tid + off < 256 ? chunk_first[tid + off] : nblk;
    __syncthreads();
    chunk_last[tid] = max(chunk_last[tid], from_left);
    chunk_first[tid] = min(chunk_first[tid], from_right);
    __syncthreads();
  }
  const int carry = tid > 0 ? chunk_last[tid - 1] : -1;
  for (int b = b0; b < b1 && rs[b] < 0; ++b) rs[b] = carry;
  const int carry_r = tid < 255 ? chunk_first[tid + 1] : nblk;
  for (int b = b1 - 1; b >= b0 && re[b] >= nblk; --b) re[b] = carry_r;
  __syncthreads();
  int32_t* l256 = tlist + kTileListHeader;
  int32_t* l192 = l256 + cap;
  int32_t* l128 = l192 + cap;
  for (int b = tid; b < nblk; b += 256) {
    if (eb[b] < 0) continue;
    const int pos = b - rs[b], len = re[b] - rs[b] + 1;
    const bool odd_tail = (len & 1) && len >= 3 && pos >= len - 3;  // the last three blocks of an odd run: two 192-row tiles
    if (odd_tail) {
      if (pos == len - 3) {
        const int at = atomicAdd(&n192, 2);
        l192[at] = 2 * b;
        l192[at + 1] = 2 * b + 3;
      }
    } else if (len == 1) {
      l128[atomicAdd(&n128, 1)] = 2 * b;
    } else if (!(pos & 1)) {
      l256[atomicAdd(&n256, 1)] = 2 * b;  // even position: first half of a 256-row tile
    }
  }
  __syncthreads();
  if (tid == 0) tlist[0] = n256, tlist[1] = n192, tlist[2] = n128;
}

__global__ void __launch_bounds__(256) contiguous_tile_list_kernel(const int32_t* m_indices, int M, int G, int32_t* tlist,
                                                                   int cap) {
  contiguous_tile_list_block(m_indices, M, G, tlist, cap);
}

// Both pre-passes of an expert-contiguous launch in one: the blocks of the scale re-layout, and one more column of
// blocks (x == tiles_x) whose first builds the tile list.  One launch less in front of the GEMM (about 5 us).
__global__ void __launch_bounds__(256) contiguous_prepass_kernel(const int32_t* m_indices, int M, int G, int32_t* tlist, int cap,
                                                                 const float* src, float* dst, int kblocks, int rows_pad,
                                                                 int64_t s_m, int64_t s_k, const int32_t* rows_map, int tiles_x) {
  if (static_cast<int>(blockIdx.x) == tiles_x) {
    if (blockIdx.y == 0) contiguous_tile_list_block(m_indices, M, G, tlist, cap);
    return;
  }
  scale_transpose_block(src, dst, M, kblocks, rows_pad, 0, s_m, s_k, rows_map, blockIdx.x, blockIdx.y, 0);
}

// First workgroup-order index of a list's tiles for this workgroup when the lists before it hold `before` tiles: the
// round robin continues where they ended.
__device__ __forceinline__ int continue_round_robin(int before) {
  const int grid = static_cast<int>(gridDim.x);
  return (static_cast<int>(blockIdx.x) + grid - before % grid) % grid;
}

}  // namespace dlb
