// Dense FP8 block-scaled GEMM between decode and prefill for gfx950: a few dozen to a few hundred rows, where a launch has
// about as many tiles as the chip has CUs.
//
// A ring kernel there spends its K step on latency, not on bytes: every step all waves meet at a barrier, then read their
// fragments at once (each operand byte several times, once per wave that needs it), then multiply; with 1 or 2 waves per
// SIMD nothing overlaps those phases.  Here the waves of a workgroup split K instead of the tile: wave w takes K blocks w,
// w + WAVES, ..., moves the operand rows of ITS block into a private piece of LDS by DMA, reads every byte back once,
// and multiplies the whole tile.  No barrier until the end: the waves drift apart and one wave's loads run under the
// others' matrix instructions.  A wave issues the DMA of its next block as soon as the fragments of the current one are in
// registers.  The partial tiles meet in LDS at the end, added in wave order.
//
// Measured (MI355X, us per launch with weights from HBM, against the ring or register-staged kernel it replaces; bench.py
// --planner-sweep wave_k): 300 x 1000 x 1040 10.9 -> 4.9 us (there in two launches), 100 x 2112 x 7168 14.5 -> 13.4 us (two
// launches), 64 x 2112 x 7168 12.9 -> 11.1 us, 300 x 4096 x 4096 20.2 -> 18.2 us, 500 x 4096 x 7168 32 -> 30 us (25.7 us with
// three sets of operands in turn, which the Infinity cache holds), 4096 x 24576 x 1040 372 -> 240 us; where the library chooses
// it, 1.10 x at 33 .. 64 rows, 1.16 x above, 1.5 x for a ragged K (geometric means; 17 .. 32 rows 0.99 x, from the caches 1.2 x).
// The bound is the DMA path of a CU (64 x 64 tiles: 16 KB per K block at 86 - 110 GB/s), and from about 10^10
// multiply-adds on the L2s (a 64 x 64 tile asks for 4 bytes per 128 of them), where the larger tiles of the ring kernels win.
// Small workgroups, so that two or more share a CU: 500 x 4096 x 7168 as 64 x 64 tiles takes 31 us with 8 waves, 26.6 with 4.
//
// Rows past M / N and bytes past a ragged K are outside the buffer descriptors' range (or sent there) and read as zero.
// Arithmetic: fp8_gemm_kernel of the reference (dlblas/kernels/fp8_gemm.py:49-60), one scale FMA per K block; the order of the
// K blocks' sums is by wave, as in the decode kernels.
#pragma once

#include "fp8_gemm_common.h"
#include "fp8_gemm_pipelined.h"
#include "fp8_gemm_stream.h"

namespace dlb {

template <int MF_, int NF_, int WAVES_>
struct WaveKCfg {
  static constexpr int MF = MF_, NF = NF_, WAVES = WAVES_;
  static constexpr int NT = WAVES * 64;
  static constexpr int BM = MF * 32, BN = NF * 32;
  static constexpr int UNITS = MF * NF * 4;                  // 16-byte accumulator units per lane
  static constexpr int WAVE_BYTES = (BM + BN) * kScaleBlock;  // one K block of both operands
  static constexpr int BUF_BYTES = WAVES * WAVE_BYTES;
  // the final sum takes as many passes as the units need to go through the buffers (a power of two: pairs stay together)
  static constexpr int PASSES = UNITS * 1024 <= WAVE_BYTES ? 1 : (UNITS * 512 <= WAVE_BYTES ? 2 : 4);
  static_assert(UNITS / PASSES * 1024 <= WAVE_BYTES && UNITS / PASSES % 2 == 0, "a pass fits the buffers");
  static constexpr int INST = (BM + BN) / 8;                  // DMA instructions per K block
  // scale table behind the buffers: BM rows of an odd pitch of at least K blocks
  static constexpr int lds_bytes(int pitch) { return BUF_BYTES + (BM * pitch * 4 + 255) / 256 * 256; }
};

template <class Cfg, bool KTAIL>
__global__ void __launch_bounds__(Cfg::NT) fp8_gemm_wavek_kernel(const Args p) {
  constexpr int MF = Cfg::MF, NF = Cfg::NF, WAVES = Cfg::WAVES, BM = Cfg::BM, BN = Cfg::BN;
  extern __shared__ __attribute__((aligned(16))) uint8_t smem[];
  const int lane = threadIdx.x & 63;
  const int wave = __builtin_amdgcn_readfirstlane(static_cast<int>(threadIdx.x >> 6));
  const int l32 = lane & 31, h = lane >> 5;
  const LaneChunks lc = make_lane_chunks(l32, h);
  const int nk = p.kblocks;
  uint8_t* buf = smem + wave * Cfg::WAVE_BYTES;
  float* table = reinterpret_cast<float*>(smem + Cfg::BUF_BYTES);

  // tile of this workgroup: consecutive tiles of an XCD form patches of up to group_m row tiles
  const int tiles = p.tiles_m * p.tiles_n;
  const int t = xcd_remap(blockIdx.x, tiles);
  const int width = p.group_m * p.tiles_n;
  const int grp = t / width, first_m = grp * p.group_m;
  const int gsz = min(p.tiles_m - first_m, p.group_m);
  const int in_grp = t - grp * width;
  const int m0 = __builtin_amdgcn_readfirstlane((first_m + in_grp % gsz) * BM);
  const int n0 = __builtin_amdgcn_readfirstlane(in_grp / gsz * BN);
  const int rows = min(BM, p.M - m0), cols = min(BN, p.N - n0);

  const uint32_t uK = static_cast<uint32_t>(p.K);
  const __amdgpu_buffer_rsrc_t a_src = make_rsrc(p.a + static_cast<int64_t>(m0) * p.K, static_cast<uint32_t>(rows) * uK);
  const __amdgpu_buffer_rsrc_t b_src = make_rsrc(p.b + static_cast<int64_t>(n0) * p.K, static_cast<uint32_t>(cols) * uK);
  // DMA instruction j of an operand fills LDS rows 8 j .. 8 j + 7; the swizzle of the 16-byte chunks depends on row & 15
  constexpr int kMaxInst = (BM > BN ? BM : BN) / 8;
  uint32_t off[kMaxInst];
#pragma unroll
  for (int j = 0; j < kMaxInst; ++j) {
    const int row = 8 * j + (lane >> 3);
    off[j] = static_cast<uint32_t>(row) * uK + static_cast<uint32_t>(((lane & 7) ^ chunk_swizzle(row)) * 16);
  }
  auto issue = [&](int kb) {
    const uint32_t koff = static_cast<uint32_t>(kb) * kScaleBlock;
    // chunks at or past the end of a ragged K: offset 2^31 is beyond the descriptor, the load returns zero
    const uint32_t left = KTAIL ? min(uK - koff, static_cast<uint32_t>(kScaleBlock)) : kScaleBlock;
    auto place = [&](int j) {
      if (!KTAIL) return off[j];
      const uint32_t chunk = static_cast<uint32_t>(((lane & 7) ^ chunk_swizzle(8 * j + (lane >> 3))) * 16);
      return chunk < left ? off[j] : 0x80000000u;
    };
#pragma unroll
    for (int j = 0; j < BN / 8; ++j) buf_dma_16<kDmaKeep>(b_src, place(j), koff, buf + BM * kScaleBlock + j * 1024);
#pragma unroll
    for (int j = 0; j < BM / 8; ++j) buf_dma_16<kDmaKeep>(a_src, place(j), koff, buf + j * 1024);
  };

  // activation scales of the tile: lanes along K, so a DMA instruction moves whole runs of a row's scales
  {
    const int pitch = p.sct_pitch;
    const float inv_pitch = 1.0f / static_cast<float>(pitch);
    const float* as = p.a_s + static_cast<int64_t>(m0) * p.as_sm;
    const int n_inst = (BM * pitch + 63) >> 6;
    for (int i = wave; i < n_inst; i += WAVES) {
      const int e = i * 64 + lane;
      const int row = static_cast<int>((static_cast<float>(e) + 0.5f) * inv_pitch);  // e / pitch, exact for e < 2^20
      const uint32_t r = static_cast<uint32_t>(min(row, rows - 1));
      const uint32_t j = static_cast<uint32_t>(min(e - row * pitch, nk - 1));
      dma_4(reinterpret_cast<const uint8_t*>(as), (r * static_cast<uint32_t>(p.as_sm) + j * static_cast<uint32_t>(p.as_sk)) * 4u,
            reinterpret_cast<uint8_t*>(table) + i * 256);
    }
  }
  int kb = wave;
  if (kb < nk) {
    issue(kb);
    wait_vmcnt<Cfg::INST>();
  } else {
    wait_vmcnt<0>();
  }
  lds_barrier();  // the whole table is there

  v16f acc[MF][NF];
#pragma unroll
  for (int mi = 0; mi < MF; ++mi)
#pragma unroll
    for (int ni = 0; ni < NF; ++ni)
#pragma unroll
      for (int u = 0; u < 16; ++u) acc[mi][ni][u] = 0.f;
  // weight scales: a tile of up to 128 columns that starts at a multiple of its width lies in one 128-block
  const const_float_ptr_t bs = (const_float_ptr_t)(p.b_s + static_cast<int64_t>(min(n0 / kScaleBlock, p.nblocks - 1)) * nk);
  float sb = bs[min(kb, nk - 1)];
  for (; kb < nk; kb += WAVES) {
    wait_vmcnt<0>();  // this wave's block has landed
    v8i x[MF][2], w[NF][2];
    float sc[MF];
#pragma unroll
    for (int ni = 0; ni < NF; ++ni) {
      w[ni][0] = lds_read_frag32(buf, (BM + ni * 32) * kScaleBlock, lc, 0);
      w[ni][1] = lds_read_frag32(buf, (BM + ni * 32) * kScaleBlock, lc, 1);
    }
#pragma unroll
    for (int mi = 0; mi < MF; ++mi) {
      x[mi][0] = lds_read_frag32(buf, mi * 32 * kScaleBlock, lc, 0);
      x[mi][1] = lds_read_frag32(buf, mi * 32 * kScaleBlock, lc, 1);
      sc[mi] = table[(mi * 32 + l32) * p.sct_pitch + kb] * sb;
    }
    asm volatile("s_waitcnt lgkmcnt(0)" ::: "memory");  // the fragments are in registers: the buffer may be refilled
    if (kb + WAVES < nk) {
      issue(kb + WAVES);
      sb = bs[kb + WAVES];
    }
#pragma unroll
    for (int mi = 0; mi < MF; ++mi)
#pragma unroll
      for (int ni = 0; ni < NF; ++ni) {
        v16f z;
#pragma unroll
        for (int u = 0; u < 16; ++u) z[u] = 0.f;
        z = mfma_32x32x64_e4m3(w[ni][0], x[mi][0], z);
        z = mfma_32x32x64_e4m3(w[ni][1], x[mi][1], z);
#pragma unroll
        for (int u = 0; u < 16; ++u) acc[mi][ni][u] = fmaf(z[u], sc[mi], acc[mi][ni][u]);
      }
  }

  // the waves' partial tiles, in wave order: unit 4 (mi NF + ni) + u = rows 32 mi + l32, columns 32 ni + 8 u + 4 h + 0..3
  constexpr int kPer = Cfg::UNITS / Cfg::PASSES;
  v4f* red = reinterpret_cast<v4f*>(smem);
#pragma unroll
  for (int pass = 0; pass < Cfg::PASSES; ++pass) {
    lds_barrier();  // every wave has read its last fragments / its sums of the pass before: the buffers are free
#pragma unroll
    for (int i = 0; i < kPer; ++i) {
      const int unit = pass * kPer + i, f = unit >> 2, u = unit & 3;
      const v16f& a = acc[f / NF][f % NF];
      red[(wave * kPer + i) * 64 + lane] = v4f{a[4 * u], a[4 * u + 1], a[4 * u + 2], a[4 * u + 3]};
    }
    lds_barrier();
    for (int q = wave; q < kPer / 2; q += WAVES) {
      v4f s[2];
#pragma unroll
      for (int i = 0; i < 2; ++i) {
        s[i] = red[(2 * q + i) * 64 + lane];
#pragma unroll
        for (int w2 = 1; w2 < WAVES; ++w2) s[i] += red[(w2 * kPer + 2 * q + i) * 64 + lane];
      }
      const int unit = pass * kPer + 2 * q, f = unit >> 2, u = unit & 3;
      const int m = f / NF * 32 + l32;
      const int n = n0 + f % NF * 32 + u * 8;
      char* c_row = static_cast<char*>(p.c) + static_cast<int64_t>(m0 + m) * p.N * (p.out_f32 ? 4 : 2);
      // lanes l and l + 32 swap halves so that each stores 8 consecutive columns
      auto row8 = [&]() __attribute__((always_inline)) {
        const v2i lo = __builtin_bit_cast(v2i, __builtin_convertvector(s[0], v4bf)), hi = __builtin_bit_cast(v2i, __builtin_convertvector(s[1], v4bf));
        const auto s0 = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(lo.x), static_cast<unsigned>(hi.x), false, false);
        const auto s1 = __builtin_amdgcn_permlane32_swap(static_cast<unsigned>(lo.y), static_cast<unsigned>(hi.y), false, false);
        return v4i{static_cast<int>(s0[0]), static_cast<int>(s1[0]), static_cast<int>(s0[1]), static_cast<int>(s1[1])};
      };
      if (p.c_whole) {  // most calls: no branch on the columns, nothing of the tails (64 x 36864 x 512 7.81 -> 7.59 us)
        const v4i v = row8();
        if (m < rows && n + 8 * h < p.N) *reinterpret_cast<v4i_el*>(reinterpret_cast<__bf16*>(c_row) + n + 8 * h) = v;
        continue;
      }
      // what the tails compute from the lane stays here: ahead of the loop over the units it held up every tile
      int eh = h;
      asm volatile("" : "+v"(eh));
      if (!p.out_f32) {
        const v4i v = row8();
        if (m < rows && n + 8 * eh < p.N) store_row8_bf16(reinterpret_cast<__bf16*>(c_row) + n + 8 * eh, v, cols == BN ? 8 : p.N - n - 8 * eh);
      } else if (m < rows) {
#pragma unroll
        for (int i = 0; i < 2; ++i) {
          const int col = n + 8 * i + 4 * eh;
          store_row4<true>(c_row, col, s[i], p.N - col);
        }
      }
    }
  }
}

}  // namespace dlb
