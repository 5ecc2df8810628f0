// C ABI of the gfx950 FP8 block-scaled GEMM library: argument validation, kernel selection, launches.
// The declarations and the contract of every entry point are in include/dlblas_fp8_gemm.h.
#include "../../include/dlblas_fp8_gemm.h"
#include "../../include/dlblas_fp8_moe.h"

#include <algorithm>
#include <atomic>
#include <cmath>
#include <cstdarg>
#include <cstdio>
#include <cstring>

#include "fp8_gemm_common.h"
#include "host_common.h"
#include "fp8_gemm_pipelined.h"
#include "fp8_gemm_ring.h"
#include "fp8_gemm_skinny.h"
#include "fp8_gemm_stream.h"
#include "fp8_gemm_tiled.h"
#include "fp8_gemm_wavek.h"
#include "fp8_quant.h"

// Scratch for dlb_fp8_gemm_noalloc: device memory that is part of the loaded code object, so a caller that cannot
// allocate (HIP graph capture, a serving loop that forbids hipMalloc) needs no workspace of its own.  Every GPU the
// library runs on holds its own copy at its own address until the process ends.  The name is only a host-side
// handle: host code uses the per-device address hipGetSymbolAddress returns (static_scratch_ptr below), never the
// name itself.
static __device__ __align__(256) unsigned char scratch[DLB_STATIC_SCRATCH_BYTES];

namespace dlb {

// ---------------------------------------------------------------------------------------------------------
// Exact path for shapes the MFMA kernels do not take (K not a multiple of 16): one thread per output
// element, e4m3 decoded in software, fp32 FMA chain per 128 block, scales applied as in
// dlblas/kernels/fp8_gemm.py:55.
// ---------------------------------------------------------------------------------------------------------
__global__ void __launch_bounds__(256) fp8_gemm_exact_kernel(const Args p) {
  const int n = blockIdx.x * 64 + (threadIdx.x & 63);
  if (n >= p.N) return;
  const uint8_t* b_row = p.b + static_cast<int64_t>(n) * p.K;
  const float* bs_row = p.b_s + static_cast<int64_t>(n / kScaleBlock) * p.kblocks;
  for (int64_t m = blockIdx.y * 4 + (threadIdx.x >> 6); m < p.M; m += static_cast<int64_t>(gridDim.y) * 4) {
    const uint8_t* a_row = p.a + m * p.K;
    const float* as_row = p.a_s + m * p.as_sm;
    float acc = 0.f;
    for (int kb = 0; kb < p.kblocks; ++kb) {
      const int k1 = min(p.K, (kb + 1) * kScaleBlock);
      float dot = 0.f;
      for (int k = kb * kScaleBlock; k < k1; ++k) dot = fmaf(e4m3_to_f32(a_row[k]), e4m3_to_f32(b_row[k]), dot);
      acc += dot * as_row[static_cast<int64_t>(kb) * p.as_sk] * bs_row[kb];
    }
    if (p.out_f32)
      static_cast<float*>(p.c)[m * p.N + n] = acc;
    else
      static_cast<__bf16*>(p.c)[m * p.N + n] = static_cast<__bf16>(acc);
  }
}

// ---------------------------------------------------------------------------------------------------------
// Host side
// ---------------------------------------------------------------------------------------------------------
thread_local char g_err[256] = "";

int fail(int code, const char* fmt, ...) {
  va_list ap;
  va_start(ap, fmt);
  vsnprintf(g_err, sizeof(g_err), fmt, ap);
  va_end(ap);
  return code;
}

void clear_error() { g_err[0] = '\0'; }

int device_cu_count(int* dev_out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<int> cached[kMaxDevices];
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return -1;
  *dev_out = dev;
  if (dev < 0 || dev >= kMaxDevices) return 256;
  int cus = cached[dev].load(std::memory_order_relaxed);
  if (cus == 0) {
    if (hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess || cus <= 0) cus = 256;
    cached[dev].store(cus, std::memory_order_relaxed);
  }
  return cus;
}

namespace {

thread_local int g_forced_variant = -1;
enum Knob : int {
  kKnobSplitK = 0,
  kKnobSkinnyWaves,
  kKnobSkinnyUnroll,
  kKnobSkinnyNFrags,
  kKnobGroupM,
  kKnobSkinnyDma,  // 0 / 1: DMA-staged decode kernel where possible, 2: register-load decode kernel
  kKnobEpilogue,   // 0 / 1: output of the pipelined kernels goes through LDS, 2: straight from registers
  kKnobSkinnyBn,   // columns per workgroup of the DMA-staged decode kernels (0 = heuristic)
  kKnobSplitKMode, // 1: K slices of the ring kernels are added inside the launch where that applies; 0 / 2: by a second launch (faster on MI355X)
  kKnobSpinLimit,  // one-launch split-K: value - 1 polls for the other slices of a tile (0 = default; 1 = none: the last arrival adds every share)
  kKnobScaleTable, // 0 / 1: row-major activation scales of the small ring kernels go through the per-tile table, 2: never
  kKnobLdsOversize,  // test hook: 1 = ask for more LDS than the GPU has, so that the launch is refused before anything is enqueued
  kKnobMaskedGrid,   // workgroups per CU of the masked layout's persistent grid (0 = default)
  kKnobTileList,     // expert-contiguous rows: 1 = device-built tile lists whenever possible, 2 = never (0 = by batch size)
  kKnobStream,       // masked layout: 1 = never the weight-streaming kernel, 2 + i = its tile shape i wherever it applies (0 = by size), 7 + i = the same, fragments read ahead
  kKnobWaveK,        // dense: 1 = never the kernel whose waves split K, 2 + i = its tile shape i wherever it applies (0 = by size)
  kKnobStreamSlices, // K slices of the weight-streaming kernel (0 = by estimate, or one where its shape is forced)
  kKnobCount
};
thread_local int g_knob[kKnobCount] = {};
// set while run() asks every kernel of the call for its launch attributes, before the first pre-pass is enqueued
thread_local bool g_prepare_only = false;
constexpr int kDefaultSpinLimit = 400;  // x about 0.5 us: far beyond the spread of the slices of one round of workgroups

enum Variant : int {
  kVarExact = 0,
  kVarTile128x128,
  kVarTile64x128,
  kVarTile128x64,
  kVarSkinny16,
  kVarSkinny32,
  kVarSkinny64,
  kVarSkinny128,
  kVarPipe256x256,
  kVarPipe128x256w8,
  kVarPipe256mix,
  kVarPipe128x128,
  kVarPipe128x64,
  kVarCount
};

const char* const kVariantNames[kVarCount] = {
    "exact", "tile128x128", "tile64x128", "tile128x64", "skinny16", "skinny32", "skinny64", "skinny128", "pipe256x256", "pipe128x256w8", "pipe256mix", "pipe128x128", "pipe128x64",
};

typedef TileCfg<128, 128, 2, 2> Tile128x128;
typedef TileCfg<64, 128, 2, 2> Tile64x128;
typedef TileCfg<128, 64, 2, 2> Tile128x64;
typedef RingCfg<4, 2, 4, 8, 2> Ring256x256;      // 8 waves, wave tile 64 x 128
typedef RingCfg<4, 2, 4, 6, 2> Ring256x192;      // narrow tiles of the mixed-width launch
typedef RingCfg<2, 4, 6, 4, 2> Ring192x256;      // wave tile 96 x 64: the two tiles of an expert's run of three 128-row blocks
typedef RingCfg<2, 4, 2, 4, 3> Ring64x256;       // wave tile 32 x 64: pieces of the tiles of a last round that is nearly empty
typedef RingCfg<2, 4, 4, 4, 3> Ring128x256;      // wave tile 64 x 64
// the same with a tile's activation scales in a table behind the ring (row-major a_s)
typedef RingCfg<4, 2, 4, 8, 2, true, 27> Ring256x256T;
typedef RingCfg<4, 2, 4, 6, 2, true, 27> Ring256x192T;
typedef RingCfg<2, 4, 4, 4, 3, true, 16> Ring128x256T;
// wave tile 32 x 64, for problems with few of the larger ones.  Eight waves instead of four with every fragment of the next step in a
// second register set (the former kernel), and a ring that runs on: us per call 1024 x 4096 x 7168 51.1 -> 44.8, 512 x 7168 x 2048 16.5
// -> 15.4, 500 x 4096 x 7168 in two slices 32.7 -> 31.6; of more than one round 3500 x 4096 x 512 26.1 -> 20.5, 2500 x 7168 x 2048 72 -> 60.
// A second register set here changes nothing (44.4): on zeros the launch takes 34 us, the rest is the clock under load.
typedef RingCfg<4, 2, 2, 4, 3> Ring128x128;
typedef RingCfg<4, 2, 2, 4, 3, true, 54> Ring128x128T;

// bytes of the three tile lists of an expert-contiguous launch over nblk 128-row blocks
constexpr size_t tile_list_bytes(int64_t nblk) {
  return (static_cast<size_t>(kTileListHeader + 3 * nblk) * sizeof(int32_t) + 255) / 256 * 256;
}
constexpr int kListLds = Ring256x256::ACT_LDS_BYTES > Ring128x256::ACT_LDS_BYTES
                             ? (Ring256x256::ACT_LDS_BYTES > Ring192x256::ACT_LDS_BYTES ? Ring256x256::ACT_LDS_BYTES : Ring192x256::ACT_LDS_BYTES)
                             : (Ring128x256::ACT_LDS_BYTES > Ring192x256::ACT_LDS_BYTES ? Ring128x256::ACT_LDS_BYTES : Ring192x256::ACT_LDS_BYTES);
// small tiles for problems with few of the large ones (M of a few hundred, or a narrow N): 4 waves, a deep ring
typedef PipeCfg<2, 2, 2, 1, 5> Pipe128x64;   // wave tile 64 x 32, 5 stages of 26 KB
// the same with the activation scales of a tile in a table behind the ring (row-major a_s; as many K blocks per
// workgroup as the LDS left by the ring holds)
typedef PipeCfg<2, 2, 2, 1, 5, true, 64> Pipe128x64T;
static_assert(Ring256x192T::LDS_BYTES <= Ring256x256T::LDS_BYTES && Ring256x192::LDS_BYTES <= Ring256x256::LDS_BYTES, "a mixed launch asks for the wide tiles' LDS");
static_assert(Pipe128x64T::LDS_BYTES <= 160 * 1024, "ring + table fit the LDS");
constexpr int kFusedMaxTiles = DLB_WS_COUNTER_BYTES / 16;  // four counter words per tile in the workspace head

// Args::c_whole.  Buffer stores need dwords; plain ones take the elements' own alignment, and c may lie on any element.
inline int whole_rows(const void* c, int64_t N, bool out_f32) {
  if (out_f32 || N % 8 != 0) return 0;
  return !misaligned(c, 4) && N < (1 << 24) ? 2 : 1;
}

// Tile shapes of the weight-streaming grouped kernel: rows x weight rows per tile, and the ring each leaves room for.
typedef StreamCfg<1, 4, 1, 2, 4, 16> Stream32x256;
typedef StreamCfg<1, 4, 2, 2, 3, 16> Stream64x256;
typedef StreamCfg<1, 4, 2, 1, 6, 16, true> Stream64x128;
typedef StreamCfg<2, 4, 2, 2, 3, 11> Stream128x256;
typedef StreamCfg<2, 2, 1, 1, 9, 16, true> Stream64x64;
// 256-column tiles with waves apart for the loads: with the quantising epilogue
typedef StreamCfg<1, 4, 1, 2, 4, 16, true> Stream32x256Apart;
typedef StreamCfg<1, 4, 2, 2, 3, 16, true> Stream64x256Apart;
enum StreamShape : int { kStreamNone = -1, kStream32x256 = 0, kStream64x256, kStream64x128, kStream128x256, kStream64x64, kStreamCount };
struct StreamDims { int bm, bn, stages, ch; };
constexpr StreamDims kStreamDims[kStreamCount] = {{32, 256, 4, 16}, {64, 256, 3, 16}, {64, 128, 6, 16}, {128, 256, 3, 11}, {64, 64, 9, 16}};

struct StreamPlan {
  int shape = kStreamNone;  // tile shape (kStreamNone: a ring kernel runs)
  int chunk_len = 0;        // K blocks per chunk of the scale table
  bool ahead = false;       // fragments read one step ahead
  int slices = 0;           // K slices of a gate/up projection, whose fp32 sums a second launch adds, activates and quantises; 0: one launch
  double us = 0.0;
};

// Tile shapes of the dense kernel whose waves split K
struct WaveKDims { int mf, nf, waves; };
constexpr WaveKDims kWaveKDims[] = {{1, 1, 8}, {1, 1, 4}, {2, 1, 8}, {1, 2, 4}, {2, 1, 4}, {2, 2, 4}, {2, 2, 2}};
constexpr int kWaveKCount = sizeof(kWaveKDims) / sizeof(kWaveKDims[0]);
constexpr int kWaveKNone = -1;

// Resident workgroups for a dense launch of `tiles` equal tiles: as many rounds as with one per CU, but even ones.  448 tiles are
// two rounds of 224 workgroups, whose clock is higher than that of 256 of which the last 64 have one tile.  A multiple of 8,
// so that a workgroup's tiles stay on one XCD.
int64_t resident_grid(int64_t tiles, int cus) {
  const int64_t even = ceil_div(ceil_div(tiles, ceil_div(tiles, cus)), 8) * 8;
  return even < cus ? even : cus;
}

// Raise a kernel's dynamic LDS limit once per (kernel, device).
template <class Kernel>
hipError_t ensure_lds(Kernel kernel, int bytes, int dev, std::atomic<unsigned long long>* done_mask) {
  if (g_knob[kKnobLdsOversize] == 1) {
    const hipError_t e =
        hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes + (1 << 20));
    if (e != hipSuccess) (void)hipGetLastError();  // the refusal is reported through the return code, not left for the caller's next HIP call
    return e;
  }
  if (bytes <= 48 * 1024) return hipSuccess;
  const unsigned long long bit = 1ull << (dev & 63);
  if (done_mask->load(std::memory_order_acquire) & bit) return hipSuccess;
  const hipError_t e =
      hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, bytes);
  if (e == hipSuccess)
    done_mask->fetch_or(bit, std::memory_order_release);
  else
    (void)hipGetLastError();
  return e;
}

template <class Cfg, int MODE>
hipError_t launch_tiled(const Args& args, int grid, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0};
  auto kernel = fp8_gemm_tiled_kernel<Cfg, MODE>;
  hipError_t e = ensure_lds(kernel, Cfg::LDS_BYTES, dev, &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, args);
  return hipGetLastError();
}

template <class Cfg>
hipError_t launch_tiled_mode(int mode, const Args& args, int grid, int dev, hipStream_t stream) {
  switch (mode) {
    case kDense:
      return launch_tiled<Cfg, kDense>(args, grid, dev, stream);
    case kContiguous:
      return launch_tiled<Cfg, kContiguous>(args, grid, dev, stream);
    default:
      return launch_tiled<Cfg, kMasked>(args, grid, dev, stream);
  }
}

template <class Cfg, int MODE>
hipError_t launch_pipelined(const Args& args, int grid, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0};
  auto kernel = fp8_gemm_pipelined_kernel<Cfg, MODE>;
  hipError_t e = ensure_lds(kernel, Cfg::LDS_BYTES, dev, &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, args);
  return hipGetLastError();
}

template <class Cfg, int MODE, bool AHEAD = false, bool ODD = false>
hipError_t launch_ring(const Args& args, int grid, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0};
  constexpr int lds = MODE == kMaskedAct ? Cfg::ACT_LDS_BYTES : Cfg::LDS_BYTES;
  auto kernel = fp8_gemm_ring_kernel<Cfg, MODE, AHEAD, ODD>;
  hipError_t e = ensure_lds(kernel, lds, dev, &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), lds, stream, args);
  return hipGetLastError();
}

// Whether a dense launch has bf16 rows off dwords, for which the 256-column tiles have kernels of their own.  us per call without / with:
// 374 x 30809 x 640 18.0 / 17.1, 1504 x 5457 x 2560 30.5 / 29.3, 2200 x 12001 x 1024 40.5 / 36.5, in 128 x 256 tiles 2683 x 10447 x 512
// 32.5 / 30.0.  Rows on dwords lose by them (374 x 30810 x 640 17.8 / 18.3) and so do 128 x 256 tiles, whose waves write 128 bytes of
// a row, at one and two K blocks (1640 x 16773 x 256 25.6 / 27.7).
inline bool odd_rows(const Args& args) { return !args.out_f32 && (args.N % 2 != 0 || misaligned(args.c, 4)) && args.splitk == 1; }

template <class Cfg>
hipError_t launch_ring_mode(int mode, const Args& args, int grid, int dev, hipStream_t stream) {
  switch (mode) {
    case kDense: {
      // resident workgroups of more than one tile: the ring that runs on (a single tile is 1 us faster without its code; the knob for
      // stores apart from the ring asks for tiles that start afresh)
      const bool ahead = args.splitk == 1 && args.c_lds && static_cast<int64_t>(args.tiles_m) * args.tiles_n > grid;
      if constexpr (Cfg::BN == 256)
        if (odd_rows(args) && (Cfg::BM == 256 || args.kblocks > 2)) return ahead ? launch_ring<Cfg, kDense, true, true>(args, grid, dev, stream) : launch_ring<Cfg, kDense, false, true>(args, grid, dev, stream);
      return ahead ? launch_ring<Cfg, kDense, true>(args, grid, dev, stream) : launch_ring<Cfg, kDense>(args, grid, dev, stream);
    }
    case kContiguous:
      if constexpr (Cfg::BM == kScaleBlock) return launch_ring<Cfg, kContiguous>(args, grid, dev, stream);  // taller tiles come from the lists
      return hipErrorInvalidValue;
    default:
      return launch_ring<Cfg, kMasked, true>(args, grid, dev, stream);
  }
}

template <class Cfg, bool KTAIL>
hipError_t launch_wavek_cfg(const Args& args, int grid, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0};
  auto kernel = fp8_gemm_wavek_kernel<Cfg, KTAIL>;
  hipError_t e = ensure_lds(kernel, 160 * 1024, dev, &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), Cfg::lds_bytes(args.sct_pitch), stream, args);
  return hipGetLastError();
}

template <bool KTAIL>
hipError_t launch_wavek(int shape, const Args& args, int grid, int dev, hipStream_t stream) {
  switch (shape) {
    case 0: return launch_wavek_cfg<WaveKCfg<1, 1, 8>, KTAIL>(args, grid, dev, stream);
    case 1: return launch_wavek_cfg<WaveKCfg<1, 1, 4>, KTAIL>(args, grid, dev, stream);
    case 2: return launch_wavek_cfg<WaveKCfg<2, 1, 8>, KTAIL>(args, grid, dev, stream);
    case 3: return launch_wavek_cfg<WaveKCfg<1, 2, 4>, KTAIL>(args, grid, dev, stream);
    case 4: return launch_wavek_cfg<WaveKCfg<2, 1, 4>, KTAIL>(args, grid, dev, stream);
    case 5: return launch_wavek_cfg<WaveKCfg<2, 2, 4>, KTAIL>(args, grid, dev, stream);
    case 6: return launch_wavek_cfg<WaveKCfg<2, 2, 2>, KTAIL>(args, grid, dev, stream);
    default: return hipErrorInvalidValue;
  }
}

template <class Cfg, int EPI, bool GATHER, bool AHEAD>
hipError_t launch_stream(const Args& args, int grid, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0};
  auto kernel = fp8_gemm_stream_kernel<Cfg, EPI, GATHER, AHEAD>;
  hipError_t e = ensure_lds(kernel, Cfg::LDS_BYTES, dev, &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), Cfg::LDS_BYTES, stream, args);
  return hipGetLastError();
}

// ahead: fragments read one step ahead of their use (plain product, tiles of 64 rows or more)
template <int EPI, bool GATHER>
hipError_t launch_stream_shape(int shape, bool ahead, const Args& args, int grid, int dev, hipStream_t stream) {
  if constexpr (EPI == kStoreProduct || EPI == kStoreSlice) {
    if (ahead) switch (shape) {
      case kStream64x256: return launch_stream<Stream64x256, EPI, GATHER, true>(args, grid, dev, stream);
      case kStream64x128: return launch_stream<Stream64x128, EPI, GATHER, true>(args, grid, dev, stream);
      case kStream128x256: return launch_stream<Stream128x256, EPI, GATHER, true>(args, grid, dev, stream);
      case kStream64x64: return launch_stream<Stream64x64, EPI, GATHER, true>(args, grid, dev, stream);
      default: break;
    }
    switch (shape) {
      case kStream64x128: return launch_stream<Stream64x128, EPI, GATHER, false>(args, grid, dev, stream);
      case kStream64x64: return launch_stream<Stream64x64, EPI, GATHER, false>(args, grid, dev, stream);
      default: break;
    }
  }
  constexpr bool act = EPI == kSiluQuant || EPI == kSiluQuantMasked;
  typedef std::conditional_t<act, Stream32x256Apart, Stream32x256> Low;
  typedef std::conditional_t<act, Stream64x256Apart, Stream64x256> High;
  switch (shape) {
    case kStream32x256: return launch_stream<Low, EPI, GATHER, false>(args, grid, dev, stream);
    case kStream64x256: return launch_stream<High, EPI, GATHER, false>(args, grid, dev, stream);
    case kStream128x256: return launch_stream<Stream128x256, EPI, GATHER, false>(args, grid, dev, stream);
    default: return hipErrorInvalidValue;
  }
}

// One call of the weight-streaming kernel and, with K slices (of a gate/up projection), of the kernel that adds them.  worst_mtiles: row tiles at most, over all
// experts; span: rows that cover nearly every expert; all_rows: of the output.
hipError_t launch_stream_plan(const StreamPlan& sp, int epi, Args ar, int64_t worst_mtiles, int64_t span, int64_t all_rows, int cus, int dev, hipStream_t stream) {
  const bool sliced = sp.slices > 0;
  const bool fused = epi != kStoreProduct && !sliced;
  ar.chunk_len = sp.chunk_len;
  ar.splitk = sliced ? sp.slices : 1;
  ar.kb_per_split = ar.kblocks / ar.splitk;
  ar.tiles_n = static_cast<int>(fused ? ar.N / 256 : ceil_div(ar.N, kStreamDims[sp.shape].bn));
  const int64_t worst = static_cast<int64_t>(ar.tiles_n) * worst_mtiles * ar.splitk;
  const int grid = static_cast<int>(ceil_div(worst < cus ? worst : cus, 32) * 32);  // tiles are dealt to the XCDs four at a time
  const Args out = ar;
  if (sliced) {
    ar.c = ar.ws;
    ar.c_gs = all_rows * ar.N;
  }
  hipError_t e;
  if (fused && epi == kSiluQuantMasked)
    e = launch_stream_shape<kSiluQuantMasked, false>(sp.shape, false, ar, grid, dev, stream);
  else if (fused)
    e = ar.a_rows ? launch_stream_shape<kSiluQuant, true>(sp.shape, false, ar, grid, dev, stream) : launch_stream_shape<kSiluQuant, false>(sp.shape, false, ar, grid, dev, stream);
  else if (sliced)
    e = ar.a_rows ? launch_stream_shape<kStoreSlice, true>(sp.shape, sp.ahead, ar, grid, dev, stream) : launch_stream_shape<kStoreSlice, false>(sp.shape, sp.ahead, ar, grid, dev, stream);
  else
    e = launch_stream_shape<kStoreProduct, false>(sp.shape, sp.ahead, ar, grid, dev, stream);
  if (e != hipSuccess || g_prepare_only || !sliced) return e;
  Args red = out;
  red.c_gs = ar.c_gs;
  // blocks for the rows nearly every expert has; a longer expert's blocks go round again
  const int64_t blocks = std::min<int64_t>(ceil_div(span * (ar.act_cols / 8), 256), ceil_div(4096, ar.G));
  const dim3 rgrid(static_cast<unsigned>(blocks < 1 ? 1 : blocks), static_cast<unsigned>(ar.G));
  if (epi == kSiluQuantMasked)
    hipLaunchKernelGGL(fp8_stream_reduce_act_kernel<kSiluQuantMasked>, rgrid, dim3(256), 0, stream, red);
  else
    hipLaunchKernelGGL(fp8_stream_reduce_act_kernel<kSiluQuant>, rgrid, dim3(256), 0, stream, red);
  return hipGetLastError();
}

template <class Cfg>
hipError_t launch_pipelined_mode(int mode, const Args& args, int grid, int dev, hipStream_t stream) {
  switch (mode) {
    case kDense:
      return launch_pipelined<Cfg, kDense>(args, grid, dev, stream);
    case kContiguous:
      return launch_pipelined<Cfg, kContiguous>(args, grid, dev, stream);
    default:
      return launch_pipelined<Cfg, kMasked>(args, grid, dev, stream);
  }
}

template <class Cfg>
hipError_t launch_skinny_cfg(bool dma, const Args& args, int dev, hipStream_t stream) {
  static std::atomic<unsigned long long> lds_done{0}, lds_done_tail{0}, lds_done_dma{0};
  const bool ktail = args.K % kScaleBlock != 0;
  // full-line DMA staging where it fits in LDS and K has no ragged block; else the register-load kernel
  if (dma && !ktail && Cfg::DMA_LDS_BYTES <= 160 * 1024 && g_knob[kKnobSkinnyDma] != 2) {
    auto kernel = fp8_gemm_skinny_dma_kernel<Cfg>;
    hipError_t e = ensure_lds(kernel, Cfg::DMA_LDS_BYTES, dev, &lds_done_dma);
    if (e != hipSuccess || g_prepare_only) return e;
    const unsigned grid = static_cast<unsigned>(ceil_div(args.N, args.sk_bn));  // its own column split, see pick_skinny_bn
    hipLaunchKernelGGL(kernel, dim3(grid), dim3(Cfg::NT), Cfg::DMA_LDS_BYTES, stream, args);
    return hipGetLastError();
  }
  auto kernel = ktail ? fp8_gemm_skinny_kernel<Cfg, true> : fp8_gemm_skinny_kernel<Cfg, false>;
  hipError_t e = ensure_lds(kernel, Cfg::RED_BYTES, dev, ktail ? &lds_done_tail : &lds_done);
  if (e != hipSuccess || g_prepare_only) return e;
  hipLaunchKernelGGL(kernel, dim3(args.tiles_n), dim3(Cfg::NT), Cfg::RED_BYTES, stream, args);
  return hipGetLastError();
}

// Skinny kernel instances: MF in {1, 2}, (waves, unroll) in a small set, n fragments in {1, 2}.
template <int MF, int NFS>
hipError_t launch_skinny_wu(int waves, int unroll, bool dma, const Args& args, int dev, hipStream_t stream) {
  if (waves >= 16) {
    if (unroll >= 4) return launch_skinny_cfg<SkinnyCfg<MF, 16, 4, NFS>>(dma, args, dev, stream);
    if (unroll >= 2) return launch_skinny_cfg<SkinnyCfg<MF, 16, 2, NFS>>(dma, args, dev, stream);
    return launch_skinny_cfg<SkinnyCfg<MF, 16, 1, NFS>>(dma, args, dev, stream);
  }
  if (waves >= 8) {
    if (unroll >= 4) return launch_skinny_cfg<SkinnyCfg<MF, 8, 4, NFS>>(dma, args, dev, stream);
    if (unroll >= 2) return launch_skinny_cfg<SkinnyCfg<MF, 8, 2, NFS>>(dma, args, dev, stream);
    return launch_skinny_cfg<SkinnyCfg<MF, 8, 1, NFS>>(dma, args, dev, stream);
  }
  if (unroll >= 4) return launch_skinny_cfg<SkinnyCfg<MF, 4, 4, NFS>>(dma, args, dev, stream);
  return launch_skinny_cfg<SkinnyCfg<MF, 4, 2, NFS>>(dma, args, dev, stream);
}

// Large activation blocks (M up to 64 / 128) keep to one K block in flight per wave: their fragments fill the registers.
template <int MF, int NFS>
hipError_t launch_skinny_big(int waves, bool dma, const Args& args, int dev, hipStream_t stream) {
  if (waves >= 16) return launch_skinny_cfg<SkinnyCfg<MF, 16, 1, NFS>>(dma, args, dev, stream);
  if (waves >= 8) return launch_skinny_cfg<SkinnyCfg<MF, 8, 1, NFS>>(dma, args, dev, stream);
  return launch_skinny_cfg<SkinnyCfg<MF, 4, 1, NFS>>(dma, args, dev, stream);
}

hipError_t launch_skinny(int mf, int nfs, int waves, int unroll, bool dma, const Args& args, int dev, hipStream_t stream) {
  switch (mf) {
    case 1:
      return nfs == 2 ? launch_skinny_wu<1, 2>(waves, unroll, dma, args, dev, stream)
                      : launch_skinny_wu<1, 1>(waves, unroll, dma, args, dev, stream);
    case 2:
      return nfs == 2 ? launch_skinny_wu<2, 2>(waves, unroll, dma, args, dev, stream)
                      : launch_skinny_wu<2, 1>(waves, unroll, dma, args, dev, stream);
    case 4:
      return nfs == 2 ? launch_skinny_big<4, 2>(waves, dma, args, dev, stream) : launch_skinny_big<4, 1>(waves, dma, args, dev, stream);
    default:
      return nfs == 2 ? launch_skinny_big<8, 2>(waves, dma, args, dev, stream) : launch_skinny_big<8, 1>(waves, dma, args, dev, stream);
  }
}


// Makespan (in units of one 256 x 256 tile) of `ta` tiles of cost 1 followed by `tb` tiles of cost `cb` < 1, handed
// out in order, each to the worker that becomes free first.  After the unit tiles `ra = ta % workers` workers are busy
// until qa + 1 and the others until qa = ta / workers; every later tile starts at one of the times qa + j cb (on one
// of the workers - ra early ones) or qa + 1 + j cb (on one of the ra late ones), smallest first, so the last start is
// found by merging two arithmetic sequences: a few steps per round of workgroups instead of one heap operation per tile.
double mixed_makespan(int64_t ta, int64_t tb, double cb, int workers) {
  const int64_t qa = ta / workers, ra = ta % workers;
  const int64_t n_early = workers - ra, n_late = ra;
  double end = ta > 0 ? static_cast<double>(qa + (ra > 0 ? 1 : 0)) : 0.0;
  int64_t left = tb, i = 0, j = 0;
  while (left > 0) {
    const double t_early = static_cast<double>(qa) + static_cast<double>(i) * cb;
    const double t_late = static_cast<double>(qa + 1) + static_cast<double>(j) * cb;
    const bool take_early = n_late == 0 || t_early <= t_late;
    const int64_t n = take_early ? n_early : n_late;
    const double start = take_early ? t_early : t_late;
    (take_early ? i : j) += 1;
    left -= n < left ? n : left;
    if (start + cb > end) end = start + cb;
  }
  return end;
}

// Columns [0, n_split) in 256-wide tiles, the rest in 192-wide tiles; returns n_split (== N: no narrow region).
// Cost: (N / 256 + 1) candidate cuts x a few steps per round, 1 to 8 us, no state.
// *makespan (optional): the launch's length in units of one 256-wide tile.
int64_t pick_mixed_split(int64_t M, int64_t N, int cus, double* makespan = nullptr) {
  const int64_t tm = ceil_div(M, 256);
  const double narrow_cost = 0.78;  // 192 / 256 of the work plus the fixed per-tile part
  int64_t best_split = N;
  if (tm * ceil_div(N, 256) > 16 * static_cast<int64_t>(cus)) {  // many rounds: the tail no longer matters
    if (makespan) *makespan = static_cast<double>(ceil_div(tm * ceil_div(N, 256), cus));
    return N;
  }
  const double uniform = mixed_makespan(tm * ceil_div(N, 256), 0, narrow_cost, cus);
  double best = uniform;
  for (int64_t ca = N / 256; ca >= 0; --ca) {
    const int64_t split = ca * 256;
    if (split >= N) continue;
    const double t = mixed_makespan(tm * ca, tm * ceil_div(N - split, 192), narrow_cost, cus);
    if (t < best - 1e-6 && t < 0.96 * uniform) best = t, best_split = split;  // not for less than 4 %
  }
  if (makespan) *makespan = best;
  return best_split;
}

// Tiles of 256 rows: widths mixed so that the rounds come out even, or all equal?  us on MI355X, 256 ... 4096 rows, K = 512 ... 18432:
//   - a workgroup per tile, one round: 9.6 + 1.26 K blocks, the first loads and the output of the tile included; a mixed launch of
//     several rounds: 2.1 + 9.3 + 1.52 K blocks per round;
//   - equal tiles, more than one round: resident workgroups whose ring runs on from tile to tile: 5.4 + 1.53 K blocks per round
//     and 5.8 for the launch.
// A last round that is not full costs half of a round (0.7 in a mixed launch, 0.44 in 128 x 256 tiles) plus its share of the rest: the chip is
// faster with fewer tiles.  43 launches lie within 5 % rms of that.  Results stored as they are now, which the fit was made before, the choice,
// 128-row tiles included, is 0.8 % behind the best of the three over 529 random problems of five K blocks and more (15 % at worst, 573 x 18582 x
// 768) and 1.1 to 1.5 % over the 80 of bench.py --planner-sweep wide_random (18 %, 2394 x 16192 x 640).
// Mixed tiles win where K is long and the last round short (4096 x 5248 x 4096: 104 / 113 us, 2048 x 17408 x 7168: 265 / 292),
// equal ones where the fixed part of a tile counts (3500 x 33024 x 1280: 203 / 183, 2048 x 18176 x 512: 45 / 38).
int pick_wide_variant(int64_t M, int64_t N, int kblocks, int cus, double* us = nullptr) {
  double span = 0.0;
  const int64_t split = pick_mixed_split(M, N, cus, &span);
  const bool mixed = split < N;
  const int64_t tiles = ceil_div(M, 256) * ceil_div(N, 256);
  const double rounds = static_cast<double>(tiles) / cus;
  const double equal_us = tiles <= cus ? 9.6 + 1.26 * kblocks : 5.8 + (0.49 * rounds + 0.51 * static_cast<double>(ceil_div(tiles, cus))) * (5.4 + 1.53 * kblocks);
  const double load = static_cast<double>(ceil_div(M, 256)) * (split / 256 + 0.78 * static_cast<double>(ceil_div(N - split, 192))) / cus;
  const double mixed_us = 2.1 + (0.7 * span + 0.3 * load) * (9.3 + 1.52 * kblocks);
  const bool equal = !mixed || equal_us <= mixed_us;
  if (us) *us = equal ? equal_us : mixed_us;
  return mixed && equal ? kVarPipe256x256 : kVarPipe256mix;  // without a narrow region both are the launch of equal tiles
}

// Prefill-sized dense problems: 256-row tiles (above) or 128 x 256 tiles?  Both run from the L2 at the pace of the matrix
// pipe there; a round of 128 x 256 tiles takes 2.4 + 0.94 K blocks, its ring runs on from tile to tile as well.
// The larger tile wins unless its rows are mostly padding (384 rows are two 256-row tiles but three of 128) or its tiles
// leave much of a round empty (2048 x 4096: 128 tiles of 256 x 256 on 256 CUs, but 256 tiles of 128 x 256):
// 384 x 18432 x 7168 82 -> 67 us, 2048 x 4096 x 7168 79 -> 67 us.  bf16 and fp32 results agree about it since both leave from the
// registers.  Limits of the smaller tile's estimate, in units of the larger one's:
//   - one and two K blocks, which the estimates were not fitted to: 0.9.  us per call, 128-row tiles / 256-row ones: 2504 x 29504 x 256 50.8
//     / 37.2, 3897 x 19856 x 256 52.7 / 38.4, 691 x 12248 x 256 13.1 / 11.4; behind the best over 285 random problems 2.4 % (10.7 %
//     with 1.2).  But 1.2 where its tiles are one round (1121 x 7040 x 256 9.4 / 10.7) and where they fill a good part of a second
//     beside one round of the larger ones, which are up to 8 % ahead there (2048 x 8192 x 256 15.5 / 14.5);
//   - three and four K blocks: 0.95, in launches of more than four rounds of the larger ones 1.07 (4096 x 32768 x 512 105 / 98): 0.9 % behind
//     the best over 286 problems, 1.6 % with 1.07 everywhere (928 x 26768 x 512 29.2 / 23.6, 1606 x 35392 x 384 fp32 71 / 52).
bool prefers_128_row_tiles(int64_t M, int64_t N, int kblocks, int cus, double* us = nullptr) {
  double wide_us = 0.0;
  pick_wide_variant(M, N, kblocks, cus, &wide_us);
  const int64_t tiles = ceil_div(M, 128) * ceil_div(N, 256), tall = ceil_div(M, 256) * ceil_div(N, 256);
  const double rounds = 0.56 * static_cast<double>(tiles) / cus + 0.44 * static_cast<double>(ceil_div(tiles, cus));
  const double half_us = 5.5 + rounds * (2.4 + 0.94 * kblocks);
  if (us) *us = std::min(wide_us, half_us);
  const bool few = tiles <= cus || (tall <= cus && 2 * tiles > 3 * cus);
  const double limit = kblocks <= 2 ? (few ? 1.2 : 0.9) : kblocks > 4 ? 1.0 : tall > 4 * cus ? 1.07 : 0.95;
  return half_us < limit * wide_us;
}

struct Plan {
  int variant;
  int bm, bn;
  int splitk;
  int sk_waves, sk_unroll, sk_nfrags;  // skinny kernel shape
  int sk_bn;                           // columns per workgroup of its DMA-staged form
  bool sk_dma;                         // decode kernels may use the DMA-staged form
};

void tile_dims(int variant, int* bm, int* bn) {
  switch (variant) {
    case kVarTile64x128:
      *bm = 64, *bn = 128;
      break;
    case kVarTile128x64:
      *bm = 128, *bn = 64;
      break;
    case kVarSkinny16:
      *bm = 16, *bn = 16;
      break;
    case kVarSkinny32:
      *bm = 32, *bn = 16;
      break;
    case kVarSkinny64:
      *bm = 64, *bn = 16;
      break;
    case kVarSkinny128:
      *bm = 128, *bn = 16;
      break;
    case kVarPipe128x256w8:
      *bm = 128, *bn = 256;
      break;
    case kVarPipe256x256:
    case kVarPipe256mix:
      *bm = 256, *bn = 256;
      break;
    case kVarPipe128x64:
      *bm = 128, *bn = 64;
      break;
    default:
      *bm = 128, *bn = 128;
  }
}

bool is_skinny(int v) { return v >= kVarSkinny16 && v <= kVarSkinny128; }
int skinny_rows(int v) { return 16 << (v - kVarSkinny16); }
bool is_pipelined(int v) { return v >= kVarPipe256x256 && v <= kVarPipe128x64; }

// Split count no larger than `want` whose slices hold at least two K blocks and whose fp32 partial matrices fit.
int clamp_splitk(int want, int64_t M, int64_t N, int kblocks, size_t avail) {
  int s = want > 32 ? 32 : want;
  if (s > kblocks / 2) s = kblocks / 2;
  const size_t per_split = static_cast<size_t>(M) * N * sizeof(float);
  if (per_split > 0 && static_cast<size_t>(s) * per_split > avail) s = static_cast<int>(avail / per_split);
  return s < 1 ? 1 : s;
}

// Output columns per workgroup of the DMA-staged decode kernels.  A CU streams weights at a rate of its own (about
// 1 / 256 of what the chip reaches), so the launch takes as long as its busiest CU: the split that gives every CU
// the same number of weight rows wins, e.g. 28 columns for N = 7168 on 256 CUs (256 workgroups) instead of 32 (224),
// or 12 for N = 2112 (176 workgroups) instead of 16 (132).  Every workgroup also reads all activation rows (from the
// L2, cheaper per row); several rounds of workgroups cost in proportion.  Multiples of 4 keep a lane's four output
// columns inside one workgroup and one 128-column scale block.
int pick_skinny_bn(int64_t N, int act_rows, int cus) {
  int best = 16;
  double best_cost = 0.0;
  for (int bn = 4; bn <= 32; bn += 4) {
    const int64_t wgs = ceil_div(N, bn);
    const double cost = static_cast<double>(ceil_div(wgs, cus)) * (bn + 0.4 * act_rows);
    if (bn == 4 || cost < best_cost - 1e-9) best = bn, best_cost = cost;
  }
  return best;
}

// Dense problems between decode and prefill (a few hundred rows, or more rows against a narrow weight matrix): too
// few 256 x 256 tiles to fill the chip, and weight rows that come from HBM because only one or two row tiles use
// them.  There a K step of a DMA-ring kernel lasts about (latency of HBM under load) / (stages in flight), whatever
// the tile size, so the estimate below is: launches + rounds of workgroups x (fixed part of a tile + K steps x time
// per step) + the second pass when K is split.  Constants measured on MI355X (microseconds; bytes per microsecond) with four-wave
// 128 x 128 tiles and 32 x 32 x 64 MFMA in all of them.
struct MidChoice {
  int variant, splitk;
  double us;
};

constexpr int64_t kRelayoutMinRows = 128;  // dense / grouped launches with more rows re-lay row-major activation scales first

MidChoice pick_mid_plan(int64_t M, int64_t N, int kblocks, int cus, size_t ws_avail) {
  struct Cand { int variant, bm, bn; double step_us; };
  static const Cand cands[] = {{kVarPipe128x256w8, 128, 256, 0.85}, {kVarPipe128x128, 128, 128, 0.65}, {kVarPipe128x64, 128, 64, 0.50}};
  const double launch = 2.6, relayout = M > kRelayoutMinRows ? 2.3 : 0.5, tile_fixed = 2.5, second_pass = 2.5, ws_rate = 3.5e6;
  // scales fetched in place (no re-layout pass): one more line request per row and K step
  const double scattered = M > kRelayoutMinRows ? 1.0 : 1.0 + 0.25 * static_cast<double>(M) / 128.0;
  MidChoice best{kVarPipe128x256w8, 1, 1e30};
  const double out_bytes = static_cast<double>(M) * N * sizeof(float);
  // fewer rows than the 128 of a tile: the clamped rows repeat lines that are already on their way
  const double short_rows = M >= 128 ? 1.0 : 0.6 + 0.4 * static_cast<double>(M) / 128.0;
  for (const Cand& c : cands) {
    for (int want : {1, 2, 3, 4, 5, 6, 7, 8, 10, 12, 14, 16}) {
      if (want > 1 && (kblocks / want < 4 || out_bytes * want > static_cast<double>(ws_avail))) continue;
      // more than 8 slices only while a slice keeps 8 K blocks (48 x 1024 x 16384: 17.9 -> 14.9 us with 16 slices;
      // 64 x 576 x 7168: 11.0 -> 12.1 us with 14)
      if (want > 8 && kblocks / want < 8) continue;
      const int per = static_cast<int>(ceil_div(kblocks, want));
      const int sk = static_cast<int>(ceil_div(kblocks, per));
      const int64_t units = ceil_div(M, c.bm) * ceil_div(N, c.bn) * sk;
      // a tile's scales come once, into a table in LDS, when the slice is short enough: no re-layout launch and no scattered scale
      // lines per K step
      const bool table = per <= (c.variant == kVarPipe128x64 ? Pipe128x64T::SCTAB_KB : c.variant == kVarPipe128x128 ? Ring128x128T::SCTAB_KB : Ring128x256T::SCTAB_KB);
      double us = launch + (table ? 0.0 : relayout) +
                  static_cast<double>(ceil_div(units, cus)) * (tile_fixed + per * c.step_us * short_rows * (table ? 1.0 : scattered));
      if (sk > 1) us += second_pass + (2.0 * sk + 0.5) * out_bytes / ws_rate;  // partial sums written, read back, result written
      if (us < best.us) best = MidChoice{c.variant, sk, us};
    }
  }
  return best;
}

// Estimate for the decode kernels at 33 .. 128 rows: what is larger of their workgroups each reading all activation rows from
// the L2 (about 8.5 TB/s over the chip) and of their waves' K blocks, fetched one after the other: a round of 8 blocks lasts
// 0.8 x (0.14 us + 24 ns per activation row + 40 ns per weight row of the workgroup) (measured at 33 .. 128 rows, 4 .. 28
// weight rows, K = 2048 .. 16384).
double decode_us(int64_t M, int64_t N, int64_t K, int kblocks, int cus) {
  const int bn = pick_skinny_bn(N, M <= 64 ? 64 : 128, cus);
  const int64_t wgs = ceil_div(N, bn);
  const double m_eff = M <= 64 ? static_cast<double>(M) : 0.5 * (M + 128.0);  // the 128-row kernel computes all 8 row fragments
  const double round_us = 0.14 + 0.0239 * m_eff + 0.04 * bn;
  const double chain_us = 0.8 * round_us * static_cast<double>(ceil_div(kblocks, 8)) * static_cast<double>(ceil_div(wgs, cus));
  const double l2_us = static_cast<double>(wgs) * M * K / 8.5e6;
  return 2.6 + (l2_us > chain_us ? l2_us : chain_us);
}

double masked_ring_us(int variant, int64_t M, int64_t N, int64_t K, int G, int64_t hint_rows, bool act, int cus);
double contiguous_small_us(int64_t rows, int64_t N, int64_t K, int G, int cus);
double contiguous_plain_us(int64_t rows, int64_t N, int64_t K, int G, int cus);
double contiguous_lists_us(int64_t rows, int64_t N, int64_t K, int G, int cus, bool there = false);

// dma_ok: the DMA kernels address their sources with 32-bit byte offsets from the tile's first row (up to 256 rows x K
// bytes, 512 scale rows x stride); false sends such problems to the kernels with 64-bit addressing.
// G, hint_rows (grouped layouts): experts, and the masked layout's typical rows per expert (<= 0: unknown).
// fixed_grouped: the caller needs the 128 x 256 kernel (the fused activation epilogues exist for it only).
Plan make_plan(int mode, int64_t M, int64_t N, int64_t K, int cus, size_t ws_bytes, bool dma_ok, int G = 1,
               int64_t hint_rows = -1, bool fixed_grouped = false, bool lists_there = false) {
  Plan pl{kVarTile128x128, 128, 128, 1, 4, 4, 1, 16, dma_ok};
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  const size_t ws_avail = ws_bytes > DLB_WS_COUNTER_BYTES ? ws_bytes - DLB_WS_COUNTER_BYTES : 0;
  int mid_splitk = 0;  // K slices chosen together with a DMA-ring variant
  int v = g_forced_variant;
  if (v < 0) {
    const bool whole_blocks = K > 0 && K % kScaleBlock == 0;
    if (K % 16 != 0) {
      v = kVarExact;
    } else if (mode == kDense && M <= 128) {
      // decode: stream the weights once, K split over the waves of a workgroup
      v = M <= 16 ? kVarSkinny16 : (M <= 32 ? kVarSkinny32 : (M <= 64 ? kVarSkinny64 : kVarSkinny128));
      // more than 64 rows against a narrow weight matrix: the few workgroups of the streaming kernel would each
      // re-read the whole activation matrix from L2; K split over workgroups in two passes is twice as fast there
      // (measured at M = 128: 2112 x 7168 44 -> 22 us, 4096 x 7168 45 -> 23 us; 7168 x 2048 stays: 16 vs 19 us)
      if (M > 64 && kblocks >= 32 && ceil_div(N, 128) * 2 <= cus) v = kVarTile128x128;
      if (M > 32 && whole_blocks) {
        // A K-split tile kernel wins when the weight matrix is narrow and K long (2112 x 7168: 18.3 -> 14.1 us at 64 rows,
        // 29 -> 17.4 us at 128; at 33 rows the streaming kernel stays ahead, 11.9 against 13.2 us)
        const double stream_us = decode_us(M, N, K, kblocks, cus);
        const MidChoice mid = pick_mid_plan(M, N, kblocks, cus, ws_avail);
        if (mid.us < stream_us) v = mid.variant, mid_splitk = mid.splitk;
        else v = M <= 64 ? kVarSkinny64 : kVarSkinny128;
      }
    } else if (whole_blocks && mode == kDense) {
      const int64_t t256 = ceil_div(M, 256) * ceil_div(N, 256);
      if (t256 * 2 >= cus) {
        v = prefers_128_row_tiles(M, N, kblocks, cus) ? kVarPipe128x256w8 : pick_wide_variant(M, N, kblocks, cus);
      } else {
        const MidChoice mid = pick_mid_plan(M, N, kblocks, cus, ws_avail);
        v = mid.variant, mid_splitk = mid.splitk;
      }
    } else if (whole_blocks) {
      v = kVarPipe128x256w8;  // grouped: 128-row tiles never straddle two experts / waste at most 127 masked rows
      const int64_t tn = ceil_div(N, 256);
      if (fixed_grouped || (mode == kContiguous && g_knob[kKnobTileList] == 1)) {
      } else if (mode == kContiguous) {
        // (the lists belong to the 128 x 256 variant)
        const double small_us = contiguous_small_us(M, N, K, G, cus);
        if (small_us < contiguous_plain_us(M, N, K, G, cus) && (ceil_div(M, kScaleBlock) <= G || small_us < contiguous_lists_us(M, N, K, G, cus, lists_there))) v = kVarPipe128x128;
      } else if (hint_rows > 0) {
        // masked, with the caller's hint: from 384 rows per expert on 256-row tiles, which fetch an expert's weights once per 256 rows (32
        // experts x ~520 rows x 4096 x 7168: 665 -> 573 us when they were introduced); fewer: the shape of the smallest estimate (the
        // same choice from 384 rows on is 0.03 % worse over 350 problems)
        if (hint_rows < M ? hint_rows >= 384 : M >= 384) {
          v = kVarPipe256x256;
        } else {
          double best_us = masked_ring_us(v, M, N, K, G, hint_rows, false, cus);
          for (int other : {kVarPipe128x128, kVarPipe256x256}) {
            const double us = masked_ring_us(other, M, N, K, G, hint_rows, false, cus);
            if (us < best_us) v = other, best_us = us;
          }
        }
      }
    } else {
      v = (M <= 64 && mode != kContiguous) ? kVarTile64x128 : kVarTile128x128;
    }
  }
  if (K % 16 != 0) v = kVarExact;
  if (is_pipelined(v) && (K % kScaleBlock != 0 || K == 0 || !dma_ok)) v = kVarTile128x128;  // DMA path moves whole K blocks
  if ((v == kVarPipe256x256 || v == kVarPipe256mix) && mode == kContiguous) v = kVarPipe128x256w8;
  if (v == kVarPipe256mix && mode != kDense) v = kVarPipe256x256;
  if (is_skinny(v) && (mode != kDense || M > skinny_rows(v))) v = kVarTile128x128;
  if (v == kVarExact && mode != kDense) v = kVarTile128x128;
  pl.variant = v;
  tile_dims(v, &pl.bm, &pl.bn);
  if (mode == kDense && is_pipelined(v) && mid_splitk > 1) pl.splitk = mid_splitk;
  // tuning knob: a K slice count for the dense tile kernels (twice the block count lets clamp_splitk go down to one
  // block per slice)
  const bool knob_splitk = g_knob[kKnobSplitK] > 0 && mode == kDense && v != kVarExact && !is_skinny(v) && v != kVarPipe256mix;
  if (knob_splitk) pl.splitk = clamp_splitk(g_knob[kKnobSplitK], M, N, kblocks * 2, ws_avail);
  if (mode != kDense || v == kVarExact || is_pipelined(v) || (kblocks < 2 && !is_skinny(v))) return pl;

  const int64_t tiles_n = ceil_div(N, pl.bn);
  const size_t avail = ws_bytes > DLB_WS_COUNTER_BYTES ? ws_bytes - DLB_WS_COUNTER_BYTES : 0;
  if (is_skinny(v)) {
    // K is split over the waves of a workgroup only.  Pick the wave count so that every wave has two or so K
    // blocks and the unroll so that a wave issues all of its loads before its first MFMA.
    int waves = kblocks >= 4 ? 8 : 4;  // (4 K blocks: 16 x 32768 x 512 7.4 -> 6.4 us with 8 waves, half of them without a block)
    // A long K against few rows: 16 waves keep twice the weight bytes in flight (1 x 2112 x 7168: 7.3 -> 6.0 us) - as
    // long as the workgroup's share of the weights is small (up to 16 rows of K = 7168: 16 x 4096 x 7168 8.4 -> 8.2 us,
    // 16 x 1536 x 7168 7.6 -> 6.4 us; from 20 rows on 8 waves are ahead: 16 x 7168 x 16384 21.7 -> 20.5 us) and one
    // round of workgroups covers the matrix (16 x 36864 x 7168: 55 -> 47 us with 8 waves).
    // (from 24 K blocks on for up to 8 rows: 1 x 4096 x 4096 6.0 -> 5.25 us, 1 x 3072 x 3072 4.9 -> 4.4 us)
    if (skinny_rows(v) == 16 && kblocks >= (M <= 8 ? 24 : 48) && K % kScaleBlock == 0) {
      const int bn16 = g_knob[kKnobSkinnyBn] > 0 ? g_knob[kKnobSkinnyBn] : pick_skinny_bn(N, 16, cus);
      // (a single row moves the limit up: 1 x 4608 x 7168, 20 rows of K = 7168 per workgroup, 9.4 -> 8.5 us with 16 waves)
      const int64_t share_limit = (M <= 8 ? 160 : 128) * 1024;
      if (static_cast<int64_t>(bn16) * K <= share_limit && ceil_div(N, bn16) <= cus) waves = 16;
    }
    if (g_knob[kKnobSkinnyWaves] > 0) waves = g_knob[kKnobSkinnyWaves] >= 16 ? 16 : (g_knob[kKnobSkinnyWaves] >= 8 ? 8 : 4);
    const int per_wave = static_cast<int>(ceil_div(kblocks, waves));
    // measured on MI355X: one K block in flight per wave is as good as more once eight waves share a row block
    int unroll = waves >= 8 ? 1 : (per_wave >= 3 ? 4 : 2);
    if (g_knob[kKnobSkinnyUnroll] > 0) unroll = g_knob[kKnobSkinnyUnroll];
    // two weight fragments per workgroup halve the activation re-reads, but only while the grid still covers the chip
    int nfrags = ceil_div(N, 32) * 4 >= 3 * cus ? 2 : 1;
    if (g_knob[kKnobSkinnyNFrags] > 0) nfrags = g_knob[kKnobSkinnyNFrags];
    pl.sk_waves = waves, pl.sk_unroll = unroll, pl.sk_nfrags = nfrags >= 2 ? 2 : 1;
    pl.sk_bn = 16 * pl.sk_nfrags;
    if (g_knob[kKnobSkinnyNFrags] <= 0 && K % kScaleBlock == 0) {
      pl.sk_bn = g_knob[kKnobSkinnyBn] > 0 ? g_knob[kKnobSkinnyBn] : pick_skinny_bn(N, skinny_rows(v), cus);
      if (pl.sk_bn % 4 != 0 || pl.sk_bn < 4 || pl.sk_bn > 32) pl.sk_bn = 16 * pl.sk_nfrags;
      pl.sk_nfrags = pl.sk_bn > 16 ? 2 : 1;
    }
    pl.bn = 16 * pl.sk_nfrags;
    // the reduction buffer (waves x fragments x 1 KB) has to fit the 160 KB of LDS whatever the knobs ask for
    const int frags = skinny_rows(v) / 16 * pl.sk_nfrags;
    while (pl.sk_waves > 4 && pl.sk_waves * frags * 1024 > 160 * 1024) pl.sk_waves /= 2;
  } else if (!knob_splitk) {
    // few tiles and a long K: split K over workgroups (partial sums in the workspace, second pass adds them)
    const int64_t tiles = ceil_div(M, pl.bm) * tiles_n;
    if (tiles * 2 > cus) return pl;
    pl.splitk = clamp_splitk(static_cast<int>(cus / tiles), M, N, kblocks, avail);  // one workgroup per CU: a single round
  }
  return pl;
}

// Everything the host decides about one launch, from shapes, strides and the workspace size alone: run() launches
// exactly this and dlb_fp8_gemm_plan reports it.
struct Resolved {
  Plan pl;
  int splitk, kb_per_split;  // K slices summed in a second pass (1 = none), K blocks per slice
  bool tile_list;            // expert-contiguous rows: device-built lists of 256-, 192- and 128-row tiles
  int64_t nblk;              //   128-row blocks it covers
  bool relayout;             // activation scales re-laid rows-contiguous in the workspace first
  int64_t rows_pad;          //   rows per K block of the re-laid copy
  size_t ws_used;            // bytes of the workspace's data region taken by list and scales; partial sums follow
  int64_t n_split;           // mixed-width launch: first column of the 192-wide tiles (N: uniform 256-wide tiles)
  int64_t grid;              // workgroups of the main kernel
  bool resident;             // dense launch of many rounds: one resident workgroup per CU walks the tiles
  bool sctab;                // small ring kernels: row-major activation scales through the per-tile table in LDS
  int sct_pitch;             //   floats per table row (odd)
  bool fused;                // K slices added inside the launch (counters in the workspace head), no second pass
  StreamPlan stream;         // masked layout: the weight-streaming kernel's share of the plan
  int wavek;                 // dense: tile shape of the kernel whose waves split K (kWaveKNone: another kernel)
};

int wavek_lds(const WaveKDims& d, int pitch) {
  const int bm = 32 * d.mf, bn = 32 * d.nf;
  return d.waves * (bm + bn) * kScaleBlock + (bm * pitch * 4 + 255) / 256 * 256;
}

// Which tile shape of the kernel whose waves split K runs a dense launch (kWaveKNone: none).
// Estimate of a launch: 1.8 us + what is longest of
//   - the busiest CU's workgroups: 1.5 us per round of resident ones (start, final sum) + K blocks x the time per block, which is
//     the larger of its bytes at 86 GB/s (the DMA path of a CU) and the trip of one block (0.21 us + 3.8 ns per operand row)
//     shared by the waves that are resident at once;
//   - every tile's operands from the L2s at 17 TB/s;  - the matrices from HBM at 6 TB/s.
// The estimate chooses the shape (2 - 3 % behind the best one, geometric mean; its rms error is 15 - 29 %, mostly too low where
// the weights come from HBM).  Whether the kernel runs at all depends on where the operands come from: from the caches (three
// weight matrices of up to 80 MB in turn stay in the 256 MB Infinity cache) it is ahead of the others, from HBM it may be
// behind.  Its time over theirs, caches / HBM, geometric means (bench.py --planner-sweep wave_k_random, 1500 problems of 512 ..
// 36864 weight rows and K = 512 .. 18432; the examples are from --planner-sweep wave_k, from HBM):
//   - up to 16 rows the decode kernels' 16-row fragments waste less (16 x 7168 x 2048 5.2 against 5.4 us), but very many columns
//     take them several rounds, whose waves idle while K is short.  From 24576 columns on 0.95 / 1.04 at up to 7 K blocks, 0.91 /
//     1.04 at 8 .. 11, 0.93 / 1.09 at 12 .. 16, 1.02 / 1.15 and 1.14 / 1.15 above (16 x 36864 x 7168 50.3 against 46.9 us): up to 11;
//   - 17 .. 64 rows: always.  17 .. 32 rows 0.87 / 1.06 at up to 80 MB (K < 2048 0.92 / 1.01, < 4096 0.85 / 1.10, longer 0.77 / 1.13:
//     32 x 2112 x 7168 11.5 against 9.6 us), 1.01 / 1.04 above; 33 .. 64 rows 0.76 / 0.92 and 0.97 / 1.02;
//   - more rows: at up to 80 MB where the estimates say so (0.70 / 0.80 there; 100 x 2112 x 7168 14.5 -> 13.4 us, 300 x 4096 x 4096
//     20 -> 18 us); larger matrices 1.22 / 1.25, and the estimates do not see it (128 x 7168 x 18432 49.8 against 40.3 us): never;
//   - a ragged K, for which only the register-staged kernels remain: always.  Up to 16 rows 0.78 / 1.00 at up to 80 MB and 0.70 /
//     0.74 above, 17 .. 64 rows 0.61 / 0.78, more 0.59 / 0.65 (300 x 1000 x 1040 10.9 -> 4.9 us, 4096 x 24576 x 1040 372 -> 240 us).
int pick_wavek(int64_t M, int64_t N, int64_t K, int cus, size_t ws_bytes) {
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  const int knob = g_knob[kKnobWaveK];
  if (knob == 1 || g_forced_variant >= 0 || g_knob[kKnobSplitK] > 0) return kWaveKNone;
  if (kblocks >= 1024) return kWaveKNone;  // no table of that many scales fits
  const bool ragged = K % kScaleBlock != 0;
  if (knob == 0 && !ragged && M <= 16 && (N < 24576 || kblocks > 11)) return kWaveKNone;
  if (knob == 0 && !ragged && M > 64 && static_cast<double>(N) * static_cast<double>(K) > 80e6) return kWaveKNone;
  int best = kWaveKNone;
  double best_us = 0.0;
  for (int i = 0; i < kWaveKCount; ++i) {
    const WaveKDims& d = kWaveKDims[i];
    if (knob >= 2 && i != knob - 2) continue;
    const int lds = wavek_lds(d, kblocks | 1);
    if (lds > 160 * 1024) continue;
    const double rows = 32.0 * (d.mf + d.nf);
    const double tiles = static_cast<double>(ceil_div(M, 32 * d.mf)) * static_cast<double>(ceil_div(N, 32 * d.nf));
    const double resident = std::max(1, std::min(160 * 1024 / lds, 16 / d.waves));
    const double per_cu = std::ceil(tiles / cus);
    const double slots = static_cast<double>(ceil_div(kblocks, d.waves)) * d.waves;
    const double block_us = std::max(rows * 128.0 / 88e3, (0.21 + 0.0038 * rows) / (d.waves * std::min(per_cu, resident)));
    const double cu_us = std::ceil(per_cu / resident) * 1.5 + per_cu * slots * block_us;
    const double l2_us = tiles * kblocks * rows * 128.0 / 17e6;
    const double hbm_us = (static_cast<double>(N) + static_cast<double>(M)) * static_cast<double>(K) / 6e6;
    const double us = 1.8 + std::max(cu_us, std::max(l2_us, hbm_us));
    if (best == kWaveKNone || us < best_us) best = i, best_us = us;
  }
  if (best == kWaveKNone || knob >= 2 || M <= 64 || ragged) return best;
  const size_t ws_avail = ws_bytes > DLB_WS_COUNTER_BYTES ? ws_bytes - DLB_WS_COUNTER_BYTES : 0;
  double other;
  const bool wide = M > 128 && ceil_div(M, 256) * ceil_div(N, 256) * 2 >= cus;
  if (wide && kblocks <= 4) return kWaveKNone;
  if (wide)
    prefers_128_row_tiles(M, N, kblocks, cus, &other);
  else
    other = pick_mid_plan(M, N, kblocks, cus, ws_avail).us;
  if (M <= 128) other = std::min(other, 1.3 * decode_us(M, N, K, kblocks, cus));  // (the 128-row decode kernel runs above its estimate at short K)
  // (where tiles of 256 columns fill half of the chip or more, this kernel's estimate is the lower one at short K and its time is not: 6 to 11
  // % behind them over 49 problems of one to four K blocks, 1121 x 7040 x 256 11.0 us for 9.4; 259 x 27200 x 1920 30.5 for 28.5; over 56 longer
  // ones it won none by 1 %)
  return best_us < (wide ? 0.85 : 0.95) * other ? best : kWaveKNone;
}

// K blocks per chunk of the streaming kernel's scale table: equal chunks of at most `ch` blocks, none shorter than the
// stages - 1 steps the issue side runs ahead (the table has two buffers), for tiles of kb_min and of kb_max blocks.  0: no such cut.
int stream_chunk_len(int kb_min, int kb_max, int ch, int stages) {
  auto last = [](int kb, int len) { return kb % len == 0 ? len : kb % len; };
  for (int len = static_cast<int>(ceil_div(kb_max, ceil_div(kb_max, ch))); len >= stages - 1 && len > 0; --len)
    if (last(kb_min, len) >= stages - 1 && last(kb_max, len) >= stages - 1) return len;
  return 0;
}

// Rows that cover nearly all experts: twice the caller's hint, at most the buffers' height.
int64_t stream_span(int64_t M, int64_t hint_rows) { return hint_rows > 0 && 2 * hint_rows < M ? 2 * hint_rows : M; }
// Time of a grouped launch (microseconds, fitted on MI355X: the weight-streaming kernel to 828 problems of 8 .. 32 experts x 1 .. 960 rows,
// N = 512 .. 7168, K = 384 .. 7168, the ring kernels to 233 of 16 .. 1024 slots; rms 8 - 12 % then.  The 64 x 64, 64 x 128 and quantising
// 256-column tiles of the former got waves of their own for the loads afterwards and take down to 0.75 of their estimates, the quantising
// ring the kernels of now; masked_second_look has estimates of the present kernels): `start` + rounds of tiles x (`tile` +
// K blocks x a step of `step` + `row` per activation row of the tile, but no shorter than its share of the stream of weights that
// the busy CUs draw, `rate` TB/s).  Taken over 0.92, 1 and 1.08 times the tile count, which is an estimate itself - except
// that experts of one row tile have no more than that (32 experts x 0 .. 16 rows x 1024 x 6144 in 64 x 128 tiles are one round of
// 256, never two).
struct TileCost {
  double start, tile, step, row, rate;
};
double grouped_us(const TileCost& c, double tiles, bool at_most, int kblocks, int bn, double rows, double sharing, int cus) {
  auto step = [&](double busy) { return std::max(c.step + c.row * rows, bn * 128.0 * busy / sharing / (c.rate * 1e6)); };
  double us = 0.0;
  for (double spread : {0.92, 1.0, at_most ? 1.0 : 1.08}) {
    const double full = std::floor(tiles * spread / cus), rest = tiles * spread - full * cus;
    us += full * (c.tile + kblocks * step(cus)) + (rest > 0.5 ? c.tile + kblocks * step(rest) : 0.0);
  }
  return c.start + us / 3.0;
}

// Typical experts of a grouped launch, from the buffers' height M and the caller's hint.
struct ExpertRows {
  double span;  // rows that cover nearly all experts
  double live;  // share of the experts that have a row
  ExpertRows(int64_t M, int64_t hint_rows) : span(static_cast<double>(stream_span(M, hint_rows))), live(span < static_cast<double>(M) ? 1.0 - std::exp(-0.5 * span) : 1.0) {}
  double row_tiles(int bm) const { return span <= bm ? 1.0 : 0.5 * (span / bm + 1.0); }
  double rows(int bm) const { return std::min(0.5 * span, static_cast<double>(bm)); }
  // the row tiles of long experts run in step and share the weights in the L2
  double sharing(int bm) const { return span > 192.0 ? row_tiles(bm) : 1.0; }
};

// The masked layout's ring kernel that make_plan chose (act: the 128 x 256 tiles with the quantising epilogue, whose constants are of the
// kernel before the present one).
double masked_ring_us(int variant, int64_t M, int64_t N, int64_t K, int G, int64_t hint_rows, bool act, int cus) {
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  int bm, bn;
  tile_dims(variant, &bm, &bn);
  TileCost c = {2.7248, 4.6095, 0.8149, 0.0024, 6.3341};  // 128 x 256
  if (act) c = {8.8, 0.8, 0.88, 0.0024, 6.2};
  else if (variant == kVarPipe128x128) c = {4.1558, 2.2571, 0.453, 0.0023, 5.7111};
  else if (variant == kVarPipe256x256) c = {3.1421, 6.5096, 1.0252, 0.0027, 5.7668};
  const ExpertRows e(M, hint_rows);
  const bool table = !act && kblocks <= (variant == kVarPipe128x128 ? Ring128x128T::SCTAB_KB : variant == kVarPipe256x256 ? Ring256x256T::SCTAB_KB : Ring128x256T::SCTAB_KB);
  const double tiles = G * e.live * e.row_tiles(bm) * static_cast<double>(act ? N / 256 : ceil_div(N, bn));
  return (M > kRelayoutMinRows && !table ? 3.5 : 0.0) + grouped_us(c, tiles, e.span <= bm, kblocks, bn, e.rows(bm), e.sharing(bm), cus);
}

// Tile shapes of the weight-streaming kernel: fragments read when needed / one step ahead / with the quantising epilogue
constexpr TileCost kStreamCost[kStreamCount] = {{2.9, 0.5, 0.74, 0.0048, 6.9}, {2.5, 1.9, 0.69, 0.0066, 6.9}, {4.1, 0.6, 0.42, 0.0048, 6.9}, {2.8, 1.7, 0.69, 0.0074, 6.9}, {4.2, 0.9, 0.38, 0.0016, 6.9}};
constexpr TileCost kStreamCostAhead[kStreamCount] = {{}, {3.0, 2.2, 0.71, 0.0041, 6.9}, {4.9, 1.0, 0.44, 0.0025, 6.9}, {3.4, 2.2, 0.71, 0.0058, 6.9}, {5.6, 0.8, 0.30, 0.0012, 6.9}};
constexpr TileCost kStreamCostAct[kStreamCount] = {{3.7, 0.6, 0.73, 0.0025, 6.9}, {3.6, 2.0, 0.72, 0.0044, 6.9}, {}, {5.2, 2.0, 0.70, 0.0049, 6.9}, {}};

// How the weight-streaming kernel runs a grouped launch (shape kStreamNone: it does not), from the typical rows of an expert, and
// whether it is to run at all: other_us is the estimate of the kernel that would run instead (0: none).  The choice is 2.8 % behind
// the best kernel, shape and number of slices (geometric mean of 75 random problems, bench.py --planner-sweep stream_random; 30 %
// at worst, gate/up of 8 experts x ~57 rows x 2560 x 2944).  With the kernels that these estimates were fitted to it was 2.3 %; a limit on
// the experts' rows in its place was 6.6 % behind for the plain product and 10.9 % with the quantising epilogue.
// With the quantising epilogue a launch may also run in two: the plain product of every (tile, K slice) first, in any tile shape, then
// the slices' sum with the activation and the quantiser.  That pays where 256-column tiles leave most CUs idle (it costs 3.8 us +
// the partial sums' way there and back): 8 experts x ~15 rows x 1792 x 3584 24.9 -> 17.0 us, 32 x ~9 x 512 x 5632 36.9 -> 22.4 us.
// The plain product gains nothing from slices that smaller tiles do not give it (1.001 x over 195 problems).
// max_slices: 1 where the bits have to be those of the steps apart (one slice changes nothing about the sums), up to kMaxStreamSlices
// inside an expert MLP.  all_rows: rows of the partial sums' matrices; slice_floats: room for them.
StreamPlan pick_stream(int64_t M, int64_t N, int64_t K, int G, int64_t hint_rows, bool act, int cus, int max_slices, int64_t all_rows, size_t slice_floats,
                       double other_us, bool by_estimates = false) {
  StreamPlan best;
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  const int knob = g_knob[kKnobStream], slice_knob = g_knob[kKnobStreamSlices];
  if (knob == 1 || g_forced_variant >= 0) return best;
  const ExpertRows e(M, hint_rows);
  const double part_bytes = static_cast<double>(G) * std::min(0.5 * e.span, static_cast<double>(M)) * static_cast<double>(N) * 4.0;
  auto offer = [&](int shape, bool ahead, bool fused_act, int slices) {
    const StreamDims& d = kStreamDims[shape];
    const int parts = slices > 0 ? slices : 1;
    const int kb_min = kblocks / parts, kb_max = static_cast<int>(ceil_div(kblocks, parts));
    if (kb_min < d.stages) return;
    if (slices > 0 && static_cast<double>(slices) * static_cast<double>(all_rows) * static_cast<double>(N) > static_cast<double>(slice_floats)) return;
    const int len = stream_chunk_len(kb_min, kb_max, d.ch, d.stages);
    if (len <= 0) return;
    const TileCost& c = fused_act ? kStreamCostAct[shape] : ahead ? kStreamCostAhead[shape] : kStreamCost[shape];
    const double tiles = G * e.live * e.row_tiles(d.bm) * static_cast<double>(fused_act ? N / 256 : ceil_div(N, d.bn)) * parts;
    double us = grouped_us(c, tiles, e.span <= d.bm, kb_max, d.bn, e.rows(d.bm), e.sharing(d.bm), cus);
    if (slices > 0) us += 3.8 + slices * part_bytes / 2.0e6;
    if (best.shape == kStreamNone || us < 0.98 * best.us) best.shape = shape, best.us = us, best.chunk_len = len, best.slices = slices, best.ahead = ahead;
  };
  for (int i = 0; i < kStreamCount; ++i) {
    if (knob >= 2 && i != (knob - 2) % kStreamCount) continue;
    const bool may_ahead = kStreamDims[i].bm > 32 && (knob < 2 || knob >= 2 + kStreamCount);
    const bool must_ahead = may_ahead && knob >= 2;
    if (act && kStreamDims[i].bn == 256 && slice_knob == 0) offer(i, false, true, 0);
    if (act && (knob == 0 || slice_knob > 0))
      for (int slices = std::max(slice_knob, 1); slices <= (slice_knob > 0 ? slice_knob : max_slices); ++slices) {
        if (!must_ahead) offer(i, false, false, slices);
        if (may_ahead) offer(i, true, false, slices);
      }
    if (!act && !must_ahead) offer(i, false, false, 0);
    if (!act && may_ahead) offer(i, true, false, 0);
  }
  // Longer experts go to the ring kernels unless the estimates say otherwise (a few of them, or narrow ones).  Plain product, us
  // here / there, 0 .. cap rows: 32 x 7168 x 2048 cap 256 116 / 141, cap 384 161 / 166, cap 512 210 / 205; 32 x 7168 x 1024 cap 448
  // 116 / 123; 32 x 4096 x 7168 cap 256 217 / 226, cap 384 305 / 298; 8 x 1152 x 768, ~640 rows 15.6 / 22.8; 8 x 512 x 1920, ~244
  // rows 14.4 / 20.1.  Quantising: 8 x 512 x 2176, ~137 rows 17.6 / 26.1; 32 x 2048 x 1920, ~181 rows 50 / 61.
  const bool longer = e.span > (act ? 192 : kblocks <= 24 ? 448 : 256);
  // by_estimates: the masked layout's plain product with a hint, where the estimates of both kernels decide from 64 rows on.  Over 350
  // problems 2.8 % behind the best kernel and shape, 5.1 % with the limits (from 256 slots on they cost 6.9 %).  This kernel runs
  // faster than its estimate there, most of all in launches of more than two rounds of 256 x 256 tiles: 32 x 256 x 7168 x 2048 118 us
  // for 148, the ring 126 for 121; 32 x 256 x 4096 x 7168 223 for 282, the ring 209 for 181.
  const bool many_rounds = static_cast<double>(G) * e.live * e.row_tiles(256) * static_cast<double>(ceil_div(N, 256)) > 2.0 * cus;
  by_estimates = by_estimates && e.span > 64.0;
  const double ahead = by_estimates ? (many_rounds ? 1.23 : 1.12) : 0.95;
  if ((longer || by_estimates) && knob == 0 && slice_knob == 0 && other_us > 0.0 && best.us > ahead * other_us) best.shape = kStreamNone;
  return best;
}

// Masked plain product with a hint above 32, from three K blocks on: a second look at the choice.  The estimates above know neither the
// output's bytes (of bf16 here) nor how the experts' rows vary, take half of the buffers for an expert's rows where twice the hint is more, and those of
// the streaming kernel are older than its waves apart.  These (us, fitted on MI355X to 2400 problems of 4 .. 64 experts x hints of 33 .. 640,
// rms 7 - 10 %): `start` + `expert` per expert + rounds of tiles x (`tile` + K blocks x (`step` + `row` per activation row of a tile)) + the
// weights and the output at `weights` and `out` TB/s.  Rounds are whole ones, averaged over what the tile count may come to: rows
// about the hint, as balanced routing leaves them, in buffers of more than three times it, rows evenly spread about it, as far as both ends
// of the buffer allow, in lower ones.
// Another kernel is taken where it is estimated 12 % ahead of the chosen one.  1200 problems outside the fit, beside the first choice alone:
// 1.024 x, 8 calls more than 5 % slower, 3.2 % behind the best kernel and shape instead of 5.6; at 6 % 1.031 x, 26 and 2.5 %.
// us per call, estimates that took half of the buffers for an expert's rows / these: 8 x 1664 x 7040, 603 rows of 896 126 / 82, 8 x 1408 x 6016
// fp32, 165 of 216 53 / 33, 4 x 1408 x 1792, 414 of 520 20.6 / 12.9, 16 x 640 x 512 fp32, 311 of 528 16.6 / 10.9; but 8 x 2688 x 768,
// 129 of 336 10.9 / 14.3.  Of 1500 further calls 185 take another kernel than the first choice: 1.20 x, 156 more than 5 % faster, 8 slower.
struct MaskedCost {
  double start, expert, tile, step, row, weights, out;
};
constexpr MaskedCost kMaskedStream[kStreamCount] = {
    {2.56, 0, 0.257, 0.334, 0.0129, 14.3, 4.05}, {3.01, 0, 0.663, 0.786, 0.00198, 25.4, 4.52}, {2.94, 0.0134, 1.31, 0.303, 0.00334, 21.7, 8.72}, {3.68, 0, 0.635, 0.584, 0.00563, 22.1, 4.84}, {3.78, 0.028, 0.665, 0.28, 0.000621, 69.7, 5.23}};
constexpr MaskedCost kMaskedStreamAhead[kStreamCount] = {
    {}, {3.5, 0, 0.908, 0.674, 0.00199, 22.3, 4.19}, {2.72, 0.0167, 1.55, 0.266, 0.00376, 20, 10}, {3.79, 0, 0.977, 0.775, 0.00232, 26.4, 4.11}, {3.25, 0.0475, 0.526, 0.254, 0.0011, 43.9, 4.55}};
constexpr MaskedCost kMasked128x256 = {2.82, 0.0957, 1.34, 0.637, 0.00193, 16.4, 5.41}, kMasked128x128 = {2.59, 0.104, 1.03, 0.405, 0.00181, 19.6, 5.41}, kMasked256x256 = {3.48, 0.0875, 2.59, 0.99, 0.000923, 21.9, 5.94};

double masked_us(const MaskedCost& c, int bm, int bn, int64_t M, int64_t N, int64_t K, int G, int64_t hint_rows, int cus) {
  const double h = static_cast<double>(std::min(hint_rows, M)), weights = static_cast<double>(N) * static_cast<double>(K);
  double live = 1.0, row_tiles, spread;  // of an expert: share that has rows, row tiles; relative spread of all tiles
  if (static_cast<double>(M) > 3.0 * h) {
    const double sd = std::sqrt(h);
    live = 1.0 - std::exp(-h);
    const double sure = std::max(0.0, std::floor((h - 4.0 * sd) / bm));  // tiles of nearly every expert
    row_tiles = live + sure;
    for (double above = (sure + 1.0) * bm; above < h + 4.0 * sd; above += bm) row_tiles += 0.5 * std::erfc((above - h) / (sd * std::sqrt(2.0)));
    spread = 0.03;
  } else {
    const double lo = std::max(0.0, 2.0 * h - static_cast<double>(M)), hi = std::min(static_cast<double>(M), 2.0 * h);
    double mean = std::ceil(h / bm), square = mean * mean;
    if (hi > 64.0 * bm) {  // long experts: without the ends of the range
      mean = h / bm + 0.5, square = mean * mean + (hi - lo) * (hi - lo) / (12.0 * bm * bm);
    } else if (hi - lo >= 1.0) {
      mean = square = 0.0;
      for (double t = std::floor(lo / bm); t * bm < hi; t += 1.0) {
        const double share = (std::min(hi, (t + 1.0) * bm) - std::max(lo, t * bm)) / (hi - lo);
        mean += share * (t + 1.0), square += share * (t + 1.0) * (t + 1.0);
      }
    }
    if (lo == 0.0) live = hi / (hi + 1.0);
    row_tiles = mean * live;
    spread = std::max(0.02, std::sqrt(std::max(0.0, square - mean * mean) / G) / row_tiles);
  }
  const double tiles = G * row_tiles * static_cast<double>(ceil_div(N, bn));
  double rounds = 0.4 * std::max(1.0, std::ceil(tiles / cus));
  for (double z : {-1.2, 1.2}) rounds += 0.3 * std::max(1.0, std::ceil(tiles * (1.0 + z * spread) / cus));
  return c.start + c.expert * G + rounds * (c.tile + static_cast<double>(ceil_div(K, kScaleBlock)) * (c.step + c.row * h / row_tiles)) + live * G * weights / (c.weights * 1e6) +
         G * h * static_cast<double>(N) * 2.0 / (c.out * 1e6);
}

void masked_second_look(Plan& pl, StreamPlan& stream, int64_t M, int64_t N, int64_t K, int G, int64_t hint_rows, int cus) {
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  auto ring_us = [&](int variant) {
    int bm, bn;
    tile_dims(variant, &bm, &bn);
    const bool small = variant == kVarPipe128x128, tall = variant == kVarPipe256x256;
    const bool table = kblocks <= (small ? Ring128x128T::SCTAB_KB : tall ? Ring256x256T::SCTAB_KB : Ring128x256T::SCTAB_KB);
    return (M > kRelayoutMinRows && !table ? 3.5 : 0.0) + masked_us(small ? kMasked128x128 : tall ? kMasked256x256 : kMasked128x256, bm, bn, M, N, K, G, hint_rows, cus);
  };
  auto stream_us = [&](int shape, bool ahead) {
    return masked_us((ahead ? kMaskedStreamAhead : kMaskedStream)[shape], kStreamDims[shape].bm, kStreamDims[shape].bn, M, N, K, G, hint_rows, cus);
  };
  const bool streams = stream.shape != kStreamNone;
  double best_us = 0.88 * (streams ? stream_us(stream.shape, stream.ahead) : ring_us(pl.variant));
  for (int variant : {kVarPipe128x256w8, kVarPipe128x128, kVarPipe256x256}) {
    const double us = ring_us(variant);
    if (us >= best_us) continue;
    best_us = us;
    stream = StreamPlan{};
    pl.variant = variant;
    tile_dims(variant, &pl.bm, &pl.bn);
  }
  for (int shape = 0; shape < kStreamCount; ++shape)
    for (bool ahead : {false, true}) {
      const StreamDims& d = kStreamDims[shape];
      const int len = kblocks < d.stages || (ahead && d.bm <= 32) ? 0 : stream_chunk_len(kblocks, kblocks, d.ch, d.stages);
      if (len <= 0) continue;
      const double us = stream_us(shape, ahead);
      if (us >= best_us) continue;
      best_us = us;
      stream.shape = shape, stream.us = us, stream.chunk_len = len, stream.slices = 0, stream.ahead = ahead;
    }
}

// Expert-contiguous rows: estimates (microseconds, fitted on MI355X to 200 problems of 8 .. 32 experts x 500 .. 12000 tokens, N and K = 512 ..
// 7168; rms 8, 8 and 17 %; their choice is 0.7 % behind the best of the three there and 0.9 % on 90 others) of 128 x 128 tiles, 128 x
// 256 tiles and the lists.  Rounds of tiles x (fixed part + K blocks x the longer of a step and its share of the weights' stream, which
// neighbouring row tiles of an expert share); the lists' step grows with the rows of a tile, two blocks where an expert has them.
// us with 128 x 256 tiles / lists: 32 experts, 5888 rows, 7168 x 2048 154 / 127, 8 experts, 9344 rows, 4096 x 1280 83 / 75; 8
// experts, 1920 rows, 3840 x 6144 68 / 78.
double contiguous_rounds_us(double tiles, double tile, double step, int kblocks, double stream_us, int cus) {
  const double full = std::floor(tiles / cus), rest = tiles - full * cus;
  auto round = [&](double busy) { return tile + kblocks * std::max(step, stream_us * busy); };
  return full * round(cus) + (rest > 0.5 ? round(rest) : 0.0);
}
// blocks of a typical expert
double contiguous_run(int64_t nblk, int G) { return std::max(1.0, static_cast<double>(nblk) / static_cast<double>(std::max<int64_t>(1, std::min<int64_t>(nblk, G)))); }
double contiguous_small_us(int64_t rows, int64_t N, int64_t K, int G, int cus) {
  const int64_t nblk = ceil_div(rows, kScaleBlock);
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  return 1.5 + contiguous_rounds_us(static_cast<double>(nblk * ceil_div(N, 128)), 4.06, 0.649, kblocks, 128 * 128.0 / (std::min(contiguous_run(nblk, G), 2.0) * 4.74e6), cus);
}
double contiguous_plain_us(int64_t rows, int64_t N, int64_t K, int G, int cus) {
  const int64_t nblk = ceil_div(rows, kScaleBlock);
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  return (kblocks > Ring128x256T::SCTAB_KB ? 5.5 : 2.0) +
         contiguous_rounds_us(static_cast<double>(nblk * ceil_div(N, 256)), 5.77, 0.907, kblocks, 256 * 128.0 / (std::min(contiguous_run(nblk, G), 1.44) * 5.4e6), cus);
}
double contiguous_lists_us(int64_t rows, int64_t N, int64_t K, int G, int cus, bool there) {
  const int64_t nblk = ceil_div(rows, kScaleBlock);
  const int kblocks = static_cast<int>(ceil_div(K, kScaleBlock));
  const double tall = std::max(0.5 * static_cast<double>(nblk), static_cast<double>(std::min<int64_t>(nblk, G)));
  const double step = 0.351 + 1.196 * 0.5 * static_cast<double>(nblk) / tall;
  double us = 0.0;
  for (double spread : {0.95, 1.0, 1.05})
    us += contiguous_rounds_us(spread * tall * static_cast<double>(ceil_div(N, 256)), 9.47, step, kblocks, 256 * 128.0 / (1.294 * 5.24e6), cus) / 3.0;
  return (there ? 0.0 : 3.6) + us;  // there: the workspace holds the lists, no launch in front builds them
}

// (act: the quantising epilogue exists for the lists only)
double contiguous_us(int64_t rows, int64_t N, int64_t K, int G, bool act, int cus) {
  const double lists_us = contiguous_lists_us(rows, N, K, G, cus);
  return act ? lists_us : std::min(lists_us, std::min(contiguous_small_us(rows, N, K, G, cus), contiguous_plain_us(rows, N, K, G, cus)));
}

// How the weight-streaming kernel runs a launch on row ranges (mlp: a step of an expert MLP, whose K may be sliced).
StreamPlan ragged_stream(int64_t rows, int64_t N, int64_t K, int G, int64_t hint_rows, bool act, bool mlp, size_t ws_bytes, int cus) {
  const bool shape_ok = K > 0 && K % kScaleBlock == 0 && K < (1ll << 24) && rows < (1ll << 31) && (!act || (N % (2 * kScaleBlock) == 0 && N * K < (1ll << 32)));
  const size_t room = ws_bytes > DLB_WS_COUNTER_BYTES ? ws_bytes - DLB_WS_COUNTER_BYTES : 0;
  if (!shape_ok) return StreamPlan{};
  return pick_stream(rows, N, K, G, hint_rows, act, cus, mlp ? kMaxStreamSlices : 1, rows, room / sizeof(float), contiguous_us(rows, N, K, G, act, cus));
}

// A step of an expert MLP on expert-contiguous rows (act: the gate/up projection, N = 2 I): 1 = the weight-streaming kernel on the
// experts' row ranges, 2 = the expert-contiguous kernels on whole blocks (act: from tile lists), 0 = neither.
int expert_form(int64_t rows, int64_t N, int64_t K, int G, int64_t hint_rows, bool act, size_t ws_bytes, int cus) {
  const size_t room = ws_bytes > DLB_WS_COUNTER_BYTES ? ws_bytes - DLB_WS_COUNTER_BYTES : 0;
  const int64_t nblk = ceil_div(rows, kScaleBlock);
  const bool shape_ok = K > 0 && K % kScaleBlock == 0 && K < (1ll << 24) && rows < (1ll << 31) && (!act || (N % (2 * kScaleBlock) == 0 && N * K < (1ll << 32)));
  if (!shape_ok || g_forced_variant >= 0) return 0;
  const bool lists = g_knob[kKnobTileList] != 2 && nblk <= kTileListMaxBlocks && tile_list_bytes(nblk) <= room;
  if (ragged_stream(rows, N, K, G, hint_rows, act, true, ws_bytes, cus).shape != kStreamNone) return 1;
  return act && !lists ? 0 : 2;
}

// overlay: the kernel whose waves split K may take the launch over from the planned variant.
// fused_act: the launch is one of the gate/up GEMMs with the activation in its epilogue (their kernels take no scale table)
Resolved resolve(int mode, int64_t rows, int64_t N, int64_t K, int G, int64_t as_sm, int64_t as_sk, bool have_ws,
                 size_t ws_bytes, int cus, bool gather_scales = false, bool fused_act = false, int64_t hint_rows = -1, bool overlay = true, int max_slices = 1, bool lists_there = false) {
  Resolved r{};
  const int64_t kblocks = ceil_div(K, kScaleBlock);
  const int64_t groups = mode == kMasked ? G : 1;  // a_s is per expert only in the masked layout; contiguous rows are one matrix
  const bool dma_ok = K < (1ll << 24) && as_sm < (1ll << 21);
  const bool usable_ws = have_ws && ws_bytes > DLB_WS_COUNTER_BYTES;
  r.pl = make_plan(mode, rows, N, K, cus, usable_ws ? ws_bytes : 0, dma_ok, G, hint_rows, fused_act || gather_scales, lists_there);
  const Plan& pl = r.pl;
  r.wavek = kWaveKNone;
  // (its scale table is fetched through 32-bit byte offsets from the tile's first row; tiles have up to 64 rows)
  const bool table_near = dma_ok && as_sk < (1ll << 20) && 63 * as_sm + (kblocks - 1) * as_sk < (1ll << 30);
  if (overlay && mode == kDense && table_near && K > 0 && K % 16 == 0) r.wavek = pick_wavek(rows, N, K, cus, usable_ws ? ws_bytes : 0);
  if (r.wavek != kWaveKNone) {
    r.pl.splitk = 1;
    r.kb_per_split = static_cast<int>(kblocks);
    r.splitk = 1;
    r.n_split = N;
    r.sct_pitch = static_cast<int>(kblocks) | 1;
    r.grid = ceil_div(rows, 32 * kWaveKDims[r.wavek].mf) * ceil_div(N, 32 * kWaveKDims[r.wavek].nf);
    return r;
  }
  if (mode == kMasked && dma_ok && K % kScaleBlock == 0 && K > 0 && static_cast<int64_t>(G) * rows < (1ll << 31))
    r.stream = pick_stream(rows, N, K, G, hint_rows, fused_act, cus, max_slices, rows * G, usable_ws ? (ws_bytes - DLB_WS_COUNTER_BYTES) / sizeof(float) : 0,
                           masked_ring_us(pl.variant, rows, N, K, G, hint_rows, fused_act, cus), !fused_act && hint_rows > 0);
  if (mode == kMasked && hint_rows > 32 && rows > 64 && kblocks > 2 && !fused_act && is_pipelined(pl.variant) && static_cast<int64_t>(G) * rows < (1ll << 31) && g_forced_variant < 0 &&
      g_knob[kKnobStream] == 0 && g_knob[kKnobStreamSlices] == 0)
    masked_second_look(r.pl, r.stream, rows, N, K, G, hint_rows, cus);
  const int want = usable_ws ? pl.splitk : 1;
  r.kb_per_split = static_cast<int>(ceil_div(kblocks > 0 ? kblocks : 1, want));
  r.splitk = static_cast<int>(ceil_div(kblocks > 0 ? kblocks : 1, r.kb_per_split));  // no empty slice
  r.n_split = N;
  if (mode == kContiguous && pl.variant == kVarPipe128x256w8 && g_forced_variant < 0 && usable_ws && kblocks > 0) {
    const int64_t nblk = ceil_div(rows, kScaleBlock);
    const size_t bytes = tile_list_bytes(nblk);
    // (the fused epilogues exist for the list kernel only)
    bool worth_it = fused_act || gather_scales || g_knob[kKnobTileList] == 1;
    if (!worth_it && g_knob[kKnobTileList] != 2 && nblk > G) worth_it = contiguous_lists_us(rows, N, K, G, cus, lists_there) < contiguous_plain_us(rows, N, K, G, cus);
    if (worth_it && nblk <= kTileListMaxBlocks && DLB_WS_COUNTER_BYTES + bytes <= ws_bytes) r.tile_list = true, r.nblk = nblk, r.ws_used = bytes;
  }
  // A tile's row-major scales come once, into a table in LDS, where its K range fits what the ring leaves of the LDS: no re-layout
  // launch in front (3 - 4 us), one cache-line request per row and tile.  us per call with the pre-pass / with the table: dense
  // 1024 x 8192 x 1536 22.5 / 19.2, 4096 x 7168 x 1024 44 / 40, 2048 x 4096 x 512 15.0 / 11.6; contiguous 8 experts, 171 rows, 1408 x 2048 19.6 / 16.3, 16
  // experts, 494 rows, 3712 x 1024 22.2 / 18.3; masked 16 x 0 .. 512 x 4096 x 1024 46 / 43.  Launches of many rounds fetch a table per
  // tile and gain nothing any more from 8 K blocks on (4096 x 24576 x 1536 175 / 175), nor lose.
  auto table_fits = [&](int kb_per) {
    if (g_knob[kKnobScaleTable] == 2 || as_sm == 1 || as_sk >= (1ll << 20) || !dma_ok || r.tile_list || gather_scales || fused_act) return false;
    switch (pl.variant) {
      case kVarPipe128x64: return mode == kDense && kb_per <= Pipe128x64T::SCTAB_KB;
      case kVarPipe128x128: return kb_per <= Ring128x128T::SCTAB_KB;
      case kVarPipe128x256w8: return (mode != kMasked || g_forced_variant < 0) && kb_per <= Ring128x256T::SCTAB_KB;
      case kVarPipe256x256: case kVarPipe256mix: return kb_per <= Ring256x256T::SCTAB_KB;
      default: return false;
    }
  };
  r.sctab = r.stream.shape == kStreamNone && table_fits(r.kb_per_split);
  // gather_scales: the re-layout pass also brings the rows into the GEMM's order, so it runs whatever the strides
  if (is_pipelined(pl.variant) && usable_ws && !r.sctab && r.stream.shape == kStreamNone &&
      (gather_scales ? kblocks > 0 : as_sk == 1 && as_sm > 1 && kblocks > 1 && rows > kRelayoutMinRows)) {
    // row-major activation scales: re-lay them rows-contiguous in the workspace first (a few microseconds) so the
    // GEMM fetches 8 cache lines of scales per K step and tile instead of 256.  Up to 128 rows the extra launch costs
    // more than the scattered scale lines (64 x 2112 x 7168: 15.9 -> 14.1 us without it)
    const int64_t rows_pad = (rows + 3) / 4 * 4;
    const int64_t need = groups * kblocks * rows_pad * static_cast<int64_t>(sizeof(float));
    if (static_cast<size_t>(need) + r.ws_used + DLB_WS_COUNTER_BYTES <= ws_bytes && rows_pad * kblocks < (1ll << 31)) {
      r.relayout = true, r.rows_pad = rows_pad;
      r.ws_used += (static_cast<size_t>(need) + 255) / 256 * 256;
    }
  }
  if (r.splitk > 1 && is_pipelined(pl.variant)) {
    // One launch: the workgroups of a tile add its slices themselves.  Needs a single round of workgroups (they wait
    // for each other, for a bounded time), a counter slot per tile and at most 32 slices (one claim bit each).
    const int64_t tiles = ceil_div(rows, pl.bm) * ceil_div(N, pl.bn);
    // Opt-in: on MI355X the device-scope round trips of that hand-over (stores out, counter, loads back) cost about
    // 3 us more than ending the launch and starting a reduction kernel behind it.
    r.fused = mode == kDense && g_knob[kKnobSplitKMode] == 1 && tiles <= kFusedMaxTiles && r.splitk <= 32 && tiles * r.splitk <= cus;
    // the partial sums of the K slices follow whatever else lives in the workspace (whole tiles in the one-launch
    // form, a [rows][N] matrix per slice otherwise); fewer slices if they do not fit
    const size_t avail = ws_bytes - DLB_WS_COUNTER_BYTES - r.ws_used;
    const size_t per_slice = r.fused ? static_cast<size_t>(tiles) * pl.bm * pl.bn * sizeof(float) : static_cast<size_t>(rows) * N * sizeof(float);
    if (per_slice * r.splitk > avail) {
      const int fit = per_slice > 0 && avail / per_slice >= 1 ? static_cast<int>(avail / per_slice) : 1;
      r.kb_per_split = static_cast<int>(ceil_div(kblocks, fit));
      r.splitk = static_cast<int>(ceil_div(kblocks, r.kb_per_split));
    }
    if (r.splitk <= 1) r.fused = false;
  }
  if (r.sctab && !table_fits(r.kb_per_split)) r.sctab = false;  // fewer, longer slices than the table holds: scales in place
  if (r.sctab)
    r.sct_pitch = r.kb_per_split | 1;
  if (pl.variant == kVarPipe256mix) r.n_split = pick_mixed_split(rows, N, cus);
  const int64_t tiles_m = ceil_div(rows, pl.bm), tiles_n = ceil_div(N, pl.bn);
  int64_t grid = tiles_m * tiles_n * r.splitk;
  if (mode == kMasked) {
    // the real tile count is only known on the device: a persistent grid
    const int64_t worst = tiles_m * tiles_n * G;
    // One resident workgroup per CU that walks its tiles: equal tiles need no balancing by the hardware's dispatcher,
    // and every further workgroup a CU has to start costs it about 2 us (32 x 256 x 7168 x 2048: 145 -> 137 us).
    const int64_t per_cu = g_knob[kKnobMaskedGrid] > 0 ? g_knob[kKnobMaskedGrid] : 1;
    grid = worst < static_cast<int64_t>(cus) * per_cu ? worst : static_cast<int64_t>(cus) * per_cu;
    grid = (grid + 31) / 32 * 32;  // the ring kernels deal tiles to the XCDs four at a time
  }
  // Dense launches of many rounds of equal tiles run one resident workgroup per CU that walks its tiles itself (the
  // ring kernels loop over tiles anyway): saves the hardware's per-workgroup start, 4 % at six rounds.  The 256-row kernel's
  // ring runs on from tile to tile, which pays from the second tile on (1 to 2 rounds 3 to 5 %, 2 to 4 rounds 7 %).
  const bool runs_on = pl.variant == kVarPipe256x256 || pl.variant == kVarPipe256mix || pl.variant == kVarPipe128x256w8 || pl.variant == kVarPipe128x128;
  const bool mixed = pl.variant == kVarPipe256mix && r.n_split < N;  // a workgroup per tile
  r.resident = mode == kDense && !mixed && grid >= (runs_on ? cus + 1ll : 4ll * cus);
  r.grid = grid;
  return r;
}

struct Problem {
  int mode;
  const void *a, *b;
  const float *a_s, *b_s;
  void* c;
  const int32_t* gidx;
  int64_t rows;  // dense: M, contiguous: M_sum, masked: M_max
  int64_t N, K;
  int G;
  int64_t as_sg, as_sm, as_sk;
  int out_dtype;
  void* ws;
  size_t ws_bytes;
  hipStream_t stream;
  // fused gate/up epilogue (dlb_fp8_gemm_grouped_{contiguous,masked}_silu_quant): c is then the e4m3 output
  // [rows][N / 2] ([G][rows][N / 2] masked)
  float* act_s = nullptr;
  int64_t act_s_sg = 0, act_s_sm = 0, act_s_sk = 0;
  // ... reading its activation rows through a table (dlb_fp8_gemm_grouped_contiguous_gather_silu_quant): row r of the
  // GEMM is row a_rows[r] of a [a_src_rows][K]; a_s has a_src_rows rows too
  const int32_t* a_rows = nullptr;
  int64_t a_src_rows = 0;
  float act_eps = 0.f;
  bool act = false;
  int64_t hint_rows = -1;  // masked layout: the caller's expected_m
  bool mlp = false;        // a step of an expert MLP: K may be sliced, and where the steps apart are faster the call is declined
  bool list_there = false;  // contiguous: the workspace still holds the tile lists of these rows
};


// Expert-contiguous rows given as one range per expert (rows the ranges leave out are not touched), on the weight-streaming
// kernel.  DLB_ERR_BAD_SHAPE, with nothing enqueued, where that kernel does not apply.
struct RaggedProblem {
  const void *a, *b;
  const float *a_s, *b_s;
  void* c;
  const int32_t *row_start, *row_end;
  const int32_t* a_rows;  // or NULL: row r is row a_rows[r] of a and a_s, which have a_src_rows rows
  int64_t a_src_rows, M_sum, N, K;
  int G;
  int64_t hint_rows, as_sm, as_sk;
  int out_dtype;
  bool act;
  float* act_s;
  int64_t act_s_sm, act_s_sk;
  float eps;
  hipStream_t stream;
  void* ws = nullptr;  // or NULL: nothing in two launches
  size_t ws_bytes = 0;
  bool mlp = false;
};

int run_ragged(const RaggedProblem& pr) {
  clear_error();
  if (pr.out_dtype != DLB_OUT_BF16 && pr.out_dtype != DLB_OUT_F32)
    return fail(DLB_ERR_BAD_DTYPE, "out_dtype %d is neither DLB_OUT_BF16 nor DLB_OUT_F32", pr.out_dtype);
  if (pr.M_sum < 0 || pr.N < 0 || pr.K < 0 || pr.G < 0 || pr.a_src_rows < 0)
    return fail(DLB_ERR_BAD_SHAPE, "negative dimension (rows=%lld N=%lld K=%lld G=%d)", (long long)pr.M_sum, (long long)pr.N, (long long)pr.K, pr.G);
  if (pr.M_sum == 0 || pr.N == 0 || pr.G == 0) return DLB_OK;
  if (!pr.a || !pr.b || !pr.a_s || !pr.b_s || !pr.c || !pr.row_start || !pr.row_end || (pr.act && !pr.act_s))
    return fail(DLB_ERR_NULL_POINTER, "a tensor pointer is NULL");
  if (pr.as_sm < 0 || pr.as_sk < 0 || (pr.act && (pr.act_s_sm < 0 || pr.act_s_sk < 0))) return fail(DLB_ERR_BAD_STRIDE, "negative scale stride");
  if (misaligned(pr.a, 16) || misaligned(pr.b, 16) || misaligned(pr.c, pr.act ? 8 : 2) || misaligned(pr.a_s, 4) || misaligned(pr.b_s, 4) ||
      (pr.act && misaligned(pr.act_s, 4)))
    return fail(DLB_ERR_ALIGNMENT, "a and b must be 16-byte aligned, c / out_q 2- / 8-byte, scales 4-byte");
  int dev = 0;
  const int cus = device_cu_count(&dev);
  if (cus < 0) return fail(DLB_ERR_LAUNCH, "hipGetDevice failed");
  const int64_t kblocks = ceil_div(pr.K, kScaleBlock);
  if (pr.ws && misaligned(pr.ws, 16)) return fail(DLB_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
  const bool usable_ws = pr.ws && pr.ws_bytes > DLB_WS_COUNTER_BYTES;
  StreamPlan sp;
  const bool fits = pr.as_sm < (1ll << 21) && pr.N < (1ll << 31) && (!pr.a_rows || (pr.act && pr.a_src_rows > 0 && pr.a_src_rows * pr.K < (1ll << 31)));
  if (fits) sp = ragged_stream(pr.M_sum, pr.N, pr.K, pr.G, pr.hint_rows, pr.act, pr.mlp, pr.ws ? pr.ws_bytes : 0, cus);
  if (sp.shape == kStreamNone)
    return fail(DLB_ERR_BAD_SHAPE, "the weight-streaming kernel does not take this problem (N=%lld K=%lld, about %lld rows per expert)",
                (long long)pr.N, (long long)pr.K, (long long)pr.hint_rows);
  Args ar;
  memset(&ar, 0, sizeof(ar));
  ar.a = static_cast<const uint8_t*>(pr.a);
  ar.b = static_cast<const uint8_t*>(pr.b);
  ar.a_s = pr.a_s;
  ar.b_s = pr.b_s;
  ar.c = pr.c;
  ar.row_start = pr.row_start;
  ar.gidx = pr.row_end;
  ar.a_rows = pr.a_rows;
  ar.a_src_rows = pr.a_src_rows;
  ar.M = static_cast<int>(pr.M_sum);
  ar.N = static_cast<int>(pr.N);
  ar.K = static_cast<int>(pr.K);
  ar.G = pr.G;
  ar.kblocks = static_cast<int>(kblocks);
  ar.nblocks = static_cast<int>(ceil_div(pr.N, kScaleBlock));
  ar.as_sm = pr.as_sm;
  ar.as_sk = pr.as_sk;
  ar.b_gs = pr.N * pr.K;
  ar.bs_gs = static_cast<int64_t>(ar.nblocks) * kblocks;
  ar.out_f32 = pr.out_dtype == DLB_OUT_F32;
  ar.act_s = pr.act_s;
  ar.act_s_sm = pr.act_s_sm;
  ar.act_s_sk = pr.act_s_sk;
  ar.act_eps = pr.eps;
  ar.act_cols = static_cast<int>(pr.N / 2);
  ar.act_q_stride = pr.N / 2;
  ar.c_whole = whole_rows(pr.c, pr.N, ar.out_f32);
  if (usable_ws) ar.ws = reinterpret_cast<float*>(static_cast<char*>(pr.ws) + DLB_WS_COUNTER_BYTES);
  const WorkspaceLock lock(pr.ws);
  const hipError_t e = launch_stream_plan(sp, pr.act ? kSiluQuant : kStoreProduct, ar, pr.G + pr.M_sum / kStreamDims[sp.shape].bm,
                                          stream_span(pr.M_sum, pr.hint_rows), pr.M_sum, cus, dev, pr.stream);
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e));
  return DLB_OK;
}

// Masked gate/up projection with the epilogue fused (rs) or the plain product and the activation apart?  Several hundred rows per
// expert: the plain product's taller tiles (32 experts x ~520 rows: 619 against 678 us).
bool steps_apart(const Resolved& rs, int64_t M, int64_t N, int G, int64_t hint_rows, int cus) {
  if (rs.stream.shape != kStreamNone || hint_rows <= 0) return false;
  const int64_t em = std::min(hint_rows, M), units = static_cast<int64_t>(G) * ceil_div(em, 128) * ceil_div(N, 256);
  return units * 2 <= cus || em >= 384 || (em >= 192 && units <= cus);
}

// Argument checks that need no device.  Returns DLB_OK with *empty set when there is nothing to compute.
int check_problem(const Problem& pr, bool* empty) {
  g_err[0] = '\0';
  *empty = false;
  if (pr.out_dtype != DLB_OUT_BF16 && pr.out_dtype != DLB_OUT_F32)
    return fail(DLB_ERR_BAD_DTYPE, "out_dtype %d is neither DLB_OUT_BF16 nor DLB_OUT_F32", pr.out_dtype);
  if (pr.rows < 0 || pr.N < 0 || pr.K < 0)
    return fail(DLB_ERR_BAD_SHAPE, "negative dimension (rows=%lld N=%lld K=%lld)", (long long)pr.rows,
                (long long)pr.N, (long long)pr.K);
  const int64_t lim = (1ll << 31) - 1024;
  if (pr.rows > lim || pr.N > lim || pr.K > lim)
    return fail(DLB_ERR_BAD_SHAPE, "dimension beyond 2^31 (rows=%lld N=%lld K=%lld)", (long long)pr.rows,
                (long long)pr.N, (long long)pr.K);
  if (pr.mode != kDense && pr.G < 0) return fail(DLB_ERR_BAD_SHAPE, "negative group count %d", pr.G);
  const int64_t groups = pr.mode == kDense ? 1 : pr.G;
  if (pr.rows == 0 || pr.N == 0 || groups == 0) {
    *empty = true;
    return DLB_OK;
  }
  if (!pr.c) return fail(DLB_ERR_NULL_POINTER, "c is NULL");
  if (pr.mode != kDense && !pr.gidx)
    return fail(DLB_ERR_NULL_POINTER, "%s is NULL", pr.mode == kContiguous ? "m_indices" : "masked_m");
  if (pr.K > 0 && (!pr.a || !pr.b || !pr.a_s || !pr.b_s))
    return fail(DLB_ERR_NULL_POINTER, "a, b, a_s or b_s is NULL");
  if (pr.mode != kDense && pr.K % 16 != 0)
    return fail(DLB_ERR_BAD_SHAPE, "grouped GEMM needs K %% 16 == 0 (K=%lld)", (long long)pr.K);
  const int64_t kblocks = ceil_div(pr.K, kScaleBlock);
  if (pr.K > 0) {
    if (pr.as_sm < 0 || pr.as_sk < 0 || pr.as_sg < 0)
      return fail(DLB_ERR_BAD_STRIDE, "negative a_s stride");
    if (pr.rows > 1 && pr.as_sm == 0) return fail(DLB_ERR_BAD_STRIDE, "a_s row stride is 0 for %lld rows", (long long)pr.rows);
    if (kblocks > 1 && pr.as_sk == 0) return fail(DLB_ERR_BAD_STRIDE, "a_s K-block stride is 0 for %lld blocks", (long long)kblocks);
    if (pr.mode == kMasked && pr.G > 1 && pr.as_sg == 0) return fail(DLB_ERR_BAD_STRIDE, "a_s group stride is 0");
  }
  const bool mfma_path = pr.K % 16 == 0;
  if (mfma_path && pr.K > 0 && (misaligned(pr.a, 16) || misaligned(pr.b, 16)))
    return fail(DLB_ERR_ALIGNMENT, "a and b must be 16-byte aligned");
  if (misaligned(pr.c, 2) || misaligned(pr.a_s, 4) || misaligned(pr.b_s, 4))
    return fail(DLB_ERR_ALIGNMENT, "c / a_s / b_s are not aligned to their element size");
  return DLB_OK;
}

int run(const Problem& pr) {
  bool empty = false;
  const int bad = check_problem(pr, &empty);
  if (bad != DLB_OK || empty) return bad;
  const WorkspaceLock lock(pr.ws);
  const int64_t groups = pr.mode == kDense ? 1 : pr.G;
  const int64_t kblocks = ceil_div(pr.K, kScaleBlock);

  int dev = 0;
  const int cus = device_cu_count(&dev);
  if (cus < 0) return fail(DLB_ERR_LAUNCH, "hipGetDevice failed");

  if (pr.ws && misaligned(pr.ws, 16)) return fail(DLB_ERR_ALIGNMENT, "workspace must be 16-byte aligned");
  const Resolved rs = resolve(pr.mode, pr.rows, pr.N, pr.K, pr.G, pr.as_sm, pr.as_sk, pr.ws != nullptr, pr.ws_bytes, cus,
                              pr.a_rows != nullptr, pr.act, pr.hint_rows, true, pr.mlp ? kMaxStreamSlices : 1, pr.list_there);
  const Plan& pl = rs.pl;
  if (pr.mlp && pr.mode == kMasked && steps_apart(rs, pr.rows, pr.N, pr.G, pr.hint_rows, cus))
    return fail(DLB_ERR_BAD_SHAPE, "GEMM, activation and quantiser apart are the faster way");
  // everything that can refuse the launch is checked before the first pre-pass kernel is enqueued
  if (rs.grid > (1ll << 30)) return fail(DLB_ERR_BAD_SHAPE, "too many tiles (%lld)", (long long)rs.grid);
  if (pl.variant == kVarExact && pr.mode != kDense) return fail(DLB_ERR_BAD_SHAPE, "exact path is dense only");
  if (pr.act) {
    // the fused epilogue exists for the tile-list kernel (contiguous) and the 128 x 256 ring kernel (masked) only:
    // whole 128-blocks of K and of the output, a workspace for the list, no forced variant; anything else is the
    // caller's cue to run the GEMM and the activation apart
    const bool kernel_ok = pr.mode == kContiguous ? rs.tile_list : pr.mode == kMasked && (rs.stream.shape != kStreamNone || pl.variant == kVarPipe128x256w8);
    if (!kernel_ok || pr.K % kScaleBlock != 0 || pr.N % (2 * kScaleBlock) != 0 || pr.N * pr.K >= (1ll << 32))
      return fail(DLB_ERR_BAD_SHAPE,
                  "fused activation needs K %% 128 == 0, N %% 256 == 0, N K < 2^32%s (N=%lld K=%lld)",
                  pr.mode == kContiguous ? " and a workspace for the tile list" : "", (long long)pr.N, (long long)pr.K);
    if (!pr.act_s || misaligned(pr.act_s, 4) || misaligned(pr.c, 8))
      return fail(DLB_ERR_ALIGNMENT, "out_s is NULL or misaligned, or out_q is not 8-byte aligned");
    if (pr.act_s_sm < 0 || pr.act_s_sk < 0 || pr.act_s_sg < 0) return fail(DLB_ERR_BAD_STRIDE, "negative out_s stride");
    if (pr.a_rows) {
      // 32-bit DMA offsets count from the first row of the source matrix; its scales are gathered by the re-layout pass
      if (pr.mode != kContiguous || !rs.relayout || pr.a_src_rows <= 0 || pr.a_src_rows * pr.K >= (1ll << 32))
        return fail(DLB_ERR_BAD_SHAPE, "gathered activation rows need a workspace for their scales and rows * K < 2^32 (rows=%lld K=%lld)",
                    (long long)pr.a_src_rows, (long long)pr.K);
      if (misaligned(pr.a_rows, 4)) return fail(DLB_ERR_ALIGNMENT, "a_row_index is misaligned");
    }
  }
  if (pl.variant == kVarExact && ceil_div(pr.N, 64) > (1ll << 31) - 1) return fail(DLB_ERR_BAD_SHAPE, "N too large for the exact path");

  Args ar;
  memset(&ar, 0, sizeof(ar));
  ar.a = static_cast<const uint8_t*>(pr.a);
  ar.b = static_cast<const uint8_t*>(pr.b);
  ar.a_s = pr.a_s;
  ar.b_s = pr.b_s;
  ar.c = pr.c;
  ar.gidx = pr.gidx;
  ar.M = static_cast<int>(pr.rows);
  ar.N = static_cast<int>(pr.N);
  ar.K = static_cast<int>(pr.K);
  ar.G = pr.mode == kDense ? 1 : pr.G;
  ar.kblocks = static_cast<int>(kblocks);
  ar.nblocks = static_cast<int>(ceil_div(pr.N, kScaleBlock));
  ar.as_sm = pr.as_sm;
  ar.as_sk = pr.as_sk;
  ar.as_gs = pr.as_sg;
  ar.a_gs = pr.rows * pr.K;
  ar.c_gs = pr.rows * pr.N;
  ar.b_gs = pr.N * pr.K;
  ar.bs_gs = static_cast<int64_t>(ar.nblocks) * kblocks;
  ar.tiles_m = static_cast<int>(ceil_div(pr.rows, pl.bm));
  ar.tiles_n = static_cast<int>(ceil_div(pr.N, pl.bn));
  ar.sk_bn = pl.sk_bn;
  ar.splitk = rs.splitk;
  ar.kb_per_split = rs.kb_per_split;
  // Row tiles per L2 patch: 8, but 7 in launches of many rounds, whose workgroups step through the patches together: us per call with 8
  // / 7 row tiles 4096 x 24576 x 1536 174 / 168, 4096 x 32768 x 512 130 / 124, 4000 x 28160 x 768 123 / 120, 3500 x 33024 x 1280
  // 191 / 186, 4096 x 24576 x 4608 447 / 446, 2048 x 36864 x 1024 99 / 100 (5 and 6 within 2 % of 7, 4 and 16 up to 11 % behind it);
  // with one to four rounds the difference is noise.
  ar.group_m = g_knob[kKnobGroupM] > 0 ? g_knob[kKnobGroupM] : (rs.resident ? 7 : 8);
  ar.out_f32 = pr.out_dtype == DLB_OUT_F32;
  ar.a_rows = pr.a_rows;
  ar.a_src_rows = pr.a_src_rows;
  ar.act_s = pr.act_s;
  ar.act_s_gs = pr.act_s_sg;
  ar.act_s_sm = pr.act_s_sm;
  ar.act_s_sk = pr.act_s_sk;
  ar.act_eps = pr.act_eps;
  ar.act_cols = static_cast<int>(pr.N / 2);
  ar.act_q_stride = pr.N / 2;
  ar.c_whole = whole_rows(pr.c, pr.N, ar.out_f32);
  ar.c_lds = g_knob[kKnobEpilogue] != 2;
  if (pr.ws && pr.ws_bytes >= DLB_WS_COUNTER_BYTES) {
    ar.ctr = static_cast<uint32_t*>(pr.ws);
    ar.ws = reinterpret_cast<float*>(static_cast<char*>(pr.ws) + DLB_WS_COUNTER_BYTES);
  }

  hipError_t e = hipSuccess;
  ar.fused_reduce = rs.fused ? 1 : 0;
  ar.spin_limit = g_knob[kKnobSpinLimit] > 0 ? g_knob[kKnobSpinLimit] - 1 : kDefaultSpinLimit;
  ar.sct_pitch = rs.sct_pitch;
  const bool tile_list = rs.tile_list;

  // The main kernel of the call.  With g_prepare_only set it only raises the kernel's dynamic-LDS limit (the one
  // step of a launch that can still fail), so that run() can do that before it enqueues the first pre-pass.
  auto main_kernel = [&]() -> hipError_t {
    if (rs.wavek == kWaveKNone) switch (pl.variant) {
      case kVarExact: {
        if (g_prepare_only) return hipSuccess;
        // rows in a grid-stride loop: the second grid dimension is limited to 65535
        const int64_t row_groups = ceil_div(pr.rows, 4);
        const dim3 grid(static_cast<unsigned>(ceil_div(pr.N, 64)), static_cast<unsigned>(row_groups < 65535 ? row_groups : 65535));
        hipLaunchKernelGGL(fp8_gemm_exact_kernel, grid, dim3(256), 0, pr.stream, ar);
        return hipGetLastError();
      }
      case kVarSkinny16:
        return launch_skinny(1, pl.sk_nfrags, pl.sk_waves, pl.sk_unroll, pl.sk_dma, ar, dev, pr.stream);
      case kVarSkinny32:
        return launch_skinny(2, pl.sk_nfrags, pl.sk_waves, pl.sk_unroll, pl.sk_dma, ar, dev, pr.stream);
      case kVarSkinny64:
        return launch_skinny(4, pl.sk_nfrags, pl.sk_waves, pl.sk_unroll, pl.sk_dma, ar, dev, pr.stream);
      case kVarSkinny128:
        return launch_skinny(8, pl.sk_nfrags, pl.sk_waves, pl.sk_unroll, pl.sk_dma, ar, dev, pr.stream);
      default:
        break;
    }
    if (rs.wavek != kWaveKNone) {
      ar.tiles_m = static_cast<int>(ceil_div(pr.rows, 32 * kWaveKDims[rs.wavek].mf));
      ar.tiles_n = static_cast<int>(ceil_div(pr.N, 32 * kWaveKDims[rs.wavek].nf));
      return pr.K % kScaleBlock != 0 ? launch_wavek<true>(rs.wavek, ar, static_cast<int>(rs.grid), dev, pr.stream)
                                     : launch_wavek<false>(rs.wavek, ar, static_cast<int>(rs.grid), dev, pr.stream);
    }
    if (rs.stream.shape != kStreamNone) {
      const int64_t worst_rows = pr.G * ceil_div(pr.rows, kStreamDims[rs.stream.shape].bm);
      return launch_stream_plan(rs.stream, pr.act ? kSiluQuantMasked : kStoreProduct, ar, worst_rows, stream_span(pr.rows, pr.hint_rows), pr.G * pr.rows,
                                cus, dev, pr.stream);
    }
    const int g = static_cast<int>(rs.grid);
    const int g_dense = static_cast<int>(rs.resident ? resident_grid(rs.grid, cus) : rs.grid);
    if (pl.variant == kVarPipe256mix) {
      const int64_t split = rs.n_split;
      if (split >= pr.N)
        return rs.sctab ? launch_ring_mode<Ring256x256T>(pr.mode, ar, g_dense, dev, pr.stream) : launch_ring_mode<Ring256x256>(pr.mode, ar, g_dense, dev, pr.stream);
      static std::atomic<unsigned long long> lds_done[4];
      const bool odd = odd_rows(ar);
      auto kernel = odd ? (rs.sctab ? fp8_gemm_ring_mixed_kernel<Ring256x256T, Ring256x192T, true> : fp8_gemm_ring_mixed_kernel<Ring256x256, Ring256x192, true>)
                        : (rs.sctab ? fp8_gemm_ring_mixed_kernel<Ring256x256T, Ring256x192T, false> : fp8_gemm_ring_mixed_kernel<Ring256x256, Ring256x192, false>);
      const int lds = rs.sctab ? Ring256x256T::LDS_BYTES : Ring256x256::LDS_BYTES;
      ar.n_split = static_cast<int>(split);
      ar.tiles_n_a = static_cast<int>(split / 256);
      ar.tiles_n_b = static_cast<int>(ceil_div(pr.N - split, 192));
      ar.tiles_a = ar.tiles_m * ar.tiles_n_a;
      const hipError_t le = ensure_lds(kernel, lds, dev, &lds_done[(rs.sctab ? 1 : 0) + (odd ? 2 : 0)]);
      if (le != hipSuccess || g_prepare_only) return le;
      hipLaunchKernelGGL(kernel, dim3(ar.tiles_a + ar.tiles_m * ar.tiles_n_b), dim3(Ring256x256::NT), lds, pr.stream, ar);
      return hipGetLastError();
    }
    if (pl.variant == kVarPipe256x256)
      return rs.sctab ? launch_ring_mode<Ring256x256T>(pr.mode, ar, g_dense, dev, pr.stream) : launch_ring_mode<Ring256x256>(pr.mode, ar, g_dense, dev, pr.stream);
    if (pl.variant == kVarPipe128x256w8 && tile_list && pr.act) {
      static std::atomic<unsigned long long> lds_done{0};
      auto kernel = fp8_gemm_ring_list_kernel<Ring256x256, Ring192x256, Ring128x256, Ring64x256, kContigListAct>;
      const hipError_t le = ensure_lds(kernel, kListLds, dev, &lds_done);
      if (le != hipSuccess || g_prepare_only) return le;
      ar.tiles_n = static_cast<int>(pr.N / 256);  // 128 output columns = 128 gate + 128 up weight rows per tile
      hipLaunchKernelGGL(kernel, dim3(cus), dim3(Ring256x256::NT), kListLds, pr.stream, ar);
      return hipGetLastError();
    }
    if (pl.variant == kVarPipe128x256w8 && tile_list) {
      static std::atomic<unsigned long long> lds_done{0};
      auto kernel = fp8_gemm_ring_list_kernel<Ring256x256, Ring192x256, Ring128x256, Ring64x256, kContigList>;
      const hipError_t le = ensure_lds(kernel, kListLds, dev, &lds_done);
      if (le != hipSuccess || g_prepare_only) return le;
      ar.tiles_n = static_cast<int>(ceil_div(pr.N, 256));
      hipLaunchKernelGGL(kernel, dim3(cus), dim3(Ring256x256::NT), kListLds, pr.stream, ar);  // one resident workgroup per CU
      return hipGetLastError();
    }
    if (pl.variant == kVarPipe128x256w8 && pr.act)
      return launch_ring<Ring128x256, kMaskedAct, true>(ar, g, dev, pr.stream);  // N / 256 column tiles, as the plain GEMM
    if (pl.variant == kVarPipe128x256w8 && rs.sctab) return launch_ring_mode<Ring128x256T>(pr.mode, ar, g_dense, dev, pr.stream);
    if (pl.variant == kVarPipe128x256w8) return launch_ring_mode<Ring128x256>(pr.mode, ar, g_dense, dev, pr.stream);
    if (pl.variant == kVarPipe128x128)
      return rs.sctab ? launch_ring_mode<Ring128x128T>(pr.mode, ar, g_dense, dev, pr.stream) : launch_ring_mode<Ring128x128>(pr.mode, ar, g_dense, dev, pr.stream);
    if (pl.variant == kVarPipe128x64)
      return rs.sctab ? launch_pipelined<Pipe128x64T, kDense>(ar, g, dev, pr.stream)
                      : launch_pipelined_mode<Pipe128x64>(pr.mode, ar, g, dev, pr.stream);
    if (pl.variant == kVarTile64x128) return launch_tiled_mode<Tile64x128>(pr.mode, ar, g, dev, pr.stream);
    if (pl.variant == kVarTile128x64) return launch_tiled_mode<Tile128x64>(pr.mode, ar, g, dev, pr.stream);
    return launch_tiled_mode<Tile128x128>(pr.mode, ar, g, dev, pr.stream);
  };
  g_prepare_only = true;
  e = main_kernel();
  g_prepare_only = false;
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "the kernel's LDS size was refused, nothing enqueued: %s", hipGetErrorString(e));

  // workspace data region: [tile list][re-laid scales][partial sums of the K slices]
  size_t ws_used = 0;
  const bool one_prepass = tile_list && rs.relayout && pr.mode == kContiguous;
  if (one_prepass) {
    // tile list and scale re-layout in one launch
    int32_t* tl = reinterpret_cast<int32_t*>(ar.ws);
    ws_used = tile_list_bytes(rs.nblk);
    float* relaid = reinterpret_cast<float*>(reinterpret_cast<char*>(ar.ws) + ws_used);
    const int tiles_x = static_cast<int>(ceil_div(rs.rows_pad, 32));
    const dim3 pgrid(static_cast<unsigned>(tiles_x + 1), static_cast<unsigned>(ceil_div(kblocks, 32)), 1);
    hipLaunchKernelGGL(contiguous_prepass_kernel, pgrid, dim3(256), 0, pr.stream, pr.gidx, static_cast<int>(pr.rows), pr.G, tl,
                       static_cast<int>(rs.nblk), pr.a_s, relaid, static_cast<int>(kblocks), static_cast<int>(rs.rows_pad), pr.as_sm,
                       pr.as_sk, pr.a_rows, tiles_x);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "pre-pass launch failed: %s", hipGetErrorString(e));
    ar.tlist = tl;
    ar.tlist_cap = static_cast<int>(rs.nblk);
    ar.a_s = relaid;
    ar.as_sm = 1;
    ar.as_sk = rs.rows_pad;
    ar.as_gs = kblocks * rs.rows_pad;
  }
  if (tile_list && !one_prepass) {
    // expert-contiguous rows: device-built lists of 256-, 192- and 128-row tiles (see contiguous_tile_list_block); they depend
    // on the rows and the experts only and lie at the same place for every N and K
    int32_t* tl = reinterpret_cast<int32_t*>(ar.ws);
    if (!pr.list_there) {
      hipLaunchKernelGGL(contiguous_tile_list_kernel, dim3(1), dim3(256), 0, pr.stream, pr.gidx, static_cast<int>(pr.rows), pr.G, tl,
                         static_cast<int>(rs.nblk));
      e = hipGetLastError();
    }
    if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "tile list launch failed: %s", hipGetErrorString(e));
    ar.tlist = tl;
    ar.tlist_cap = static_cast<int>(rs.nblk);
    ws_used = tile_list_bytes(rs.nblk);
  }
  if (rs.relayout && !one_prepass) {
    float* relaid = reinterpret_cast<float*>(reinterpret_cast<char*>(ar.ws) + ws_used);
    const dim3 tgrid(static_cast<unsigned>(ceil_div(rs.rows_pad, 32)), static_cast<unsigned>(ceil_div(kblocks, 32)),
                     static_cast<unsigned>(pr.mode == kMasked ? groups : 1));
    hipLaunchKernelGGL(fp8_scale_transpose_kernel, tgrid, dim3(256), 0, pr.stream, pr.a_s, relaid, static_cast<int>(pr.rows),
                       static_cast<int>(kblocks), static_cast<int>(rs.rows_pad), pr.mode == kMasked ? pr.as_sg : 0, pr.as_sm,
                       pr.as_sk, pr.a_rows);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "scale re-layout launch failed: %s", hipGetErrorString(e));
    ar.a_s = relaid;
    ar.as_sm = 1;
    ar.as_sk = rs.rows_pad;
    ar.as_gs = kblocks * rs.rows_pad;
  }
  if (ar.splitk > 1 && is_pipelined(pl.variant)) ar.ws = reinterpret_cast<float*>(reinterpret_cast<char*>(ar.ws) + rs.ws_used);
  e = main_kernel();
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e));
  if (ar.splitk > 1 && !rs.fused && pr.mode == kDense && pl.variant != kVarExact && !is_skinny(pl.variant)) {
    const int64_t total = pr.rows * pr.N;
    hipLaunchKernelGGL(fp8_splitk_reduce_kernel, dim3(static_cast<unsigned>(ceil_div(ceil_div(total, 4), 256))), dim3(256), 0,
                       pr.stream, ar.ws, pr.c, total, ar.splitk, ar.out_f32);
    e = hipGetLastError();
    if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "split-K reduction launch failed: %s", hipGetErrorString(e));
  }
  return DLB_OK;
}

// The slice of `scratch` that calls on `stream` work in.  The array's device address is looked up once per device
// (with that device current) and kept; a stream is bound to the first free slice of its device at its first call and
// keeps it until the process ends, so calls on different streams never share scratch memory.  More streams than slices:
// DLB_ERR_WORKSPACE.
int static_scratch_slice(hipStream_t stream, void** out) {
  constexpr int kMaxDevices = 64;
  static std::atomic<void*> ptr_of[kMaxDevices];
  static std::atomic<uintptr_t> owner[kMaxDevices][DLB_STATIC_SCRATCH_SLICES];  // 0 = free, else the stream handle + 1
  int dev = 0;
  if (hipGetDevice(&dev) != hipSuccess) return fail(DLB_ERR_LAUNCH, "hipGetDevice failed");
  if (dev < 0 || dev >= kMaxDevices) return fail(DLB_ERR_LAUNCH, "device ordinal %d beyond the %d this library tracks", dev, kMaxDevices);
  void* ptr = ptr_of[dev].load(std::memory_order_acquire);
  if (!ptr) {
    const hipError_t e = hipGetSymbolAddress(&ptr, HIP_SYMBOL(scratch));
    if (e != hipSuccess || !ptr) return fail(DLB_ERR_LAUNCH, "hipGetSymbolAddress(scratch) failed on device %d: %s", dev, hipGetErrorString(e));
    ptr_of[dev].store(ptr, std::memory_order_release);
  }
  const uintptr_t key = reinterpret_cast<uintptr_t>(stream) + 1;
  for (int i = 0; i < DLB_STATIC_SCRATCH_SLICES; ++i) {
    uintptr_t cur = owner[dev][i].load(std::memory_order_acquire);
    if (cur == 0 && owner[dev][i].compare_exchange_strong(cur, key, std::memory_order_acq_rel)) cur = key;
    if (cur == key) {
      *out = static_cast<char*>(ptr) + static_cast<size_t>(i) * DLB_STATIC_SCRATCH_SLICE_BYTES;
      return DLB_OK;
    }
  }
  return fail(DLB_ERR_WORKSPACE,
              "the %d slices of the static scratch of device %d are bound to other streams; use dlb_fp8_gemm with a workspace "
              "for this stream", DLB_STATIC_SCRATCH_SLICES, dev);
}

template <int IN>
void launch_quant_group(const QuantArgs& qa, int lanes, unsigned blocks, hipStream_t st) {
  const dim3 grid(blocks), block(256);
  switch (lanes) {
    case 1: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 1>), grid, block, 0, st, qa); break;
    case 2: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 2>), grid, block, 0, st, qa); break;
    case 4: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 4>), grid, block, 0, st, qa); break;
    case 8: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 8>), grid, block, 0, st, qa); break;
    case 16: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 16>), grid, block, 0, st, qa); break;
    case 32: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 32>), grid, block, 0, st, qa); break;
    case 64: hipLaunchKernelGGL((fp8_quant_group_kernel<IN, 64>), grid, block, 0, st, qa); break;
    default: hipLaunchKernelGGL(fp8_quant_group_generic_kernel<IN>, grid, block, 0, st, qa);
  }
}

}  // namespace
}  // namespace dlb

// ---------------------------------------------------------------------------------------------------------
// extern "C" surface
// ---------------------------------------------------------------------------------------------------------
extern "C" {

int dlb_abi_version(void) { return DLB_ABI_VERSION; }

const char* dlb_last_error(void) { return dlb::g_err; }

size_t dlb_fp8_gemm_workspace_bytes(int64_t rows, int64_t N, int64_t K) {
  (void)K;
  if (rows <= 0 || N <= 0) return DLB_WS_COUNTER_BYTES;
  // Split-K only runs while the un-split grid cannot fill the chip, so (tiles x splits) stays within a few
  // hundred fp32 tiles of at most 128 x 128: 32 MiB covers every plan; the planner lowers the split count to
  // fit whatever it is given.
  const size_t cap = static_cast<size_t>(32) << 20;
  const int64_t padded = dlb::ceil_div(rows, 128) * dlb::ceil_div(N, 128);
  const size_t want = padded > 1024 ? cap : static_cast<size_t>(padded) * 128 * 128 * sizeof(float) * 16;
  return DLB_WS_COUNTER_BYTES + (want < cap ? want : cap);
}

int dlb_workspace_lock(const void* workspace) {
  dlb::clear_error();
  if (!workspace) return dlb::fail(DLB_ERR_NULL_POINTER, "workspace is NULL");
  dlb::workspace_mutex(workspace).lock();
  return DLB_OK;
}

int dlb_workspace_unlock(const void* workspace) {
  dlb::clear_error();
  if (!workspace) return dlb::fail(DLB_ERR_NULL_POINTER, "workspace is NULL");
  dlb::workspace_mutex(workspace).unlock();
  return DLB_OK;
}

int dlb_fp8_gemm(const void* a, const void* b, const float* a_s, const float* b_s, void* c, int64_t M, int64_t N,
                 int64_t K, int64_t as_stride_m, int64_t as_stride_k, int out_dtype, void* workspace,
                 size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kDense, a, b, a_s, b_s, c, nullptr, M, N, K, 1, 0, as_stride_m, as_stride_k, out_dtype,
                  workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  return dlb::run(pr);
}

int dlb_fp8_gemm_noalloc(const void* a, const void* b, const float* a_s, const float* b_s, void* c, int64_t M, int64_t N,
                         int64_t K, int64_t as_stride_m, int64_t as_stride_k, int out_dtype, void* stream) {
  dlb::Problem pr{dlb::kDense, a, b, a_s, b_s, c, nullptr, M, N, K, 1, 0, as_stride_m, as_stride_k, out_dtype,
                  nullptr, 0, static_cast<hipStream_t>(stream)};
  bool empty = false;
  const int bad = dlb::check_problem(pr, &empty);
  if (bad != DLB_OK || empty) return bad;
  // What the plan of this problem would keep in a workspace of any size besides the partial sums of K slices (those
  // adapt to the space there is): the activation scales re-laid rows-contiguous.  That has to fit a slice.
  int dev = 0;
  const int cus = dlb::device_cu_count(&dev);
  if (cus < 0) return dlb::fail(DLB_ERR_LAUNCH, "hipGetDevice failed");
  const dlb::Resolved want = dlb::resolve(dlb::kDense, M, N, K, 1, as_stride_m, as_stride_k, true, static_cast<size_t>(1) << 40, cus);
  const size_t room = DLB_STATIC_SCRATCH_SLICE_BYTES - DLB_WS_COUNTER_BYTES;
  if (want.ws_used > room)
    return dlb::fail(DLB_ERR_WORKSPACE,
                     "M=%lld x ceil(K/128)=%lld needs %lld bytes of re-laid scales, a slice of the static scratch holds %lld; use "
                     "dlb_fp8_gemm with a workspace", (long long)M, (long long)dlb::ceil_div(K, dlb::kScaleBlock), (long long)want.ws_used,
                     (long long)room);
  void* ws = nullptr;
  const int rc = dlb::static_scratch_slice(pr.stream, &ws);
  if (rc != DLB_OK) return rc;
  pr.ws = ws;
  pr.ws_bytes = DLB_STATIC_SCRATCH_SLICE_BYTES;
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_contiguous(const void* a, const void* b, const float* a_s, const float* b_s, void* c,
                                    const int32_t* m_indices, int64_t M_sum, int64_t N, int64_t K, int32_t G,
                                    int64_t as_stride_m, int64_t as_stride_k, int out_dtype, void* workspace,
                                    size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kContiguous, a, b, a_s, b_s, c, m_indices, M_sum, N, K, G, 0, as_stride_m, as_stride_k,
                  out_dtype, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_contiguous_same_rows(const void* a, const void* b, const float* a_s, const float* b_s, void* c,
                                              const int32_t* m_indices, int64_t M_sum, int64_t N, int64_t K, int32_t G,
                                              int64_t as_stride_m, int64_t as_stride_k, int out_dtype, void* workspace,
                                              size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kContiguous, a, b, a_s, b_s, c, m_indices, M_sum, N, K, G, 0, as_stride_m, as_stride_k,
                  out_dtype, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.list_there = true;
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_contiguous_silu_quant(const void* a, const void* b, const float* a_s, const float* b_s, void* out_q,
                                               float* out_s, const int32_t* m_indices, int64_t M_sum, int64_t N, int64_t K,
                                               int32_t G, int64_t as_stride_m, int64_t as_stride_k, int64_t os_stride_m,
                                               int64_t os_stride_k, float eps, void* workspace, size_t workspace_bytes,
                                               void* stream) {
  dlb::Problem pr{dlb::kContiguous, a, b, a_s, b_s, out_q, m_indices, M_sum, N, K, G, 0, as_stride_m, as_stride_k,
                  DLB_OUT_BF16, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.act = true;
  pr.act_s = out_s;
  pr.act_s_sm = os_stride_m;
  pr.act_s_sk = os_stride_k;
  pr.act_eps = eps;
  if (M_sum > 0 && N > 0 && G > 0 && !out_s) return dlb::fail(DLB_ERR_NULL_POINTER, "out_s is NULL");
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_contiguous_gather_silu_quant(const void* a, const void* b, const float* a_s, const float* b_s,
                                                      void* out_q, float* out_s, const int32_t* m_indices,
                                                      const int32_t* a_row_index, int64_t a_rows, int64_t M_sum, int64_t N,
                                                      int64_t K, int32_t G, int64_t as_stride_m, int64_t as_stride_k,
                                                      int64_t os_stride_m, int64_t os_stride_k, float eps, void* workspace,
                                                      size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kContiguous, a, b, a_s, b_s, out_q, m_indices, M_sum, N, K, G, 0, as_stride_m, as_stride_k,
                  DLB_OUT_BF16, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.act = true;
  pr.act_s = out_s;
  pr.act_s_sm = os_stride_m;
  pr.act_s_sk = os_stride_k;
  pr.act_eps = eps;
  pr.a_rows = a_row_index;
  pr.a_src_rows = a_rows;
  if (M_sum > 0 && N > 0 && G > 0 && !out_s) return dlb::fail(DLB_ERR_NULL_POINTER, "out_s is NULL");
  if (M_sum > 0 && N > 0 && G > 0 && !a_row_index) return dlb::fail(DLB_ERR_NULL_POINTER, "a_row_index is NULL");
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_masked_silu_quant(const void* a, const void* b, const float* a_s, const float* b_s, void* out_q,
                                           float* out_s, const int32_t* masked_m, int32_t expected_m, int64_t M_max,
                                           int64_t N, int64_t K, int32_t G, int64_t as_stride_g, int64_t as_stride_m,
                                           int64_t as_stride_k, int64_t os_stride_g, int64_t os_stride_m, int64_t os_stride_k,
                                           float eps, void* workspace, size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kMasked, a, b, a_s, b_s, out_q, masked_m, M_max, N, K, G, as_stride_g, as_stride_m, as_stride_k,
                  DLB_OUT_BF16, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.act = true;
  pr.act_s = out_s;
  pr.act_s_sg = os_stride_g;
  pr.act_s_sm = os_stride_m;
  pr.act_s_sk = os_stride_k;
  pr.act_eps = eps;
  pr.hint_rows = expected_m;
  if (M_max > 0 && N > 0 && G > 0 && !out_s) return dlb::fail(DLB_ERR_NULL_POINTER, "out_s is NULL");
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_masked(const void* a, const void* b, const float* a_s, const float* b_s, void* c,
                                const int32_t* masked_m, int32_t expected_m, int64_t M_max, int64_t N, int64_t K,
                                int32_t G, int64_t as_stride_g, int64_t as_stride_m, int64_t as_stride_k,
                                int out_dtype, void* workspace, size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kMasked, a, b, a_s, b_s, c, masked_m, M_max, N, K, G, as_stride_g, as_stride_m, as_stride_k,
                  out_dtype, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.hint_rows = expected_m;
  return dlb::run(pr);
}

int dlb_fp8_gemm_grouped_ragged(const void* a, const void* b, const float* a_s, const float* b_s, void* c, const int32_t* row_start,
                                const int32_t* row_end, int32_t expected_m, int64_t M_sum, int64_t N, int64_t K, int32_t G,
                                int64_t as_stride_m, int64_t as_stride_k, int out_dtype, void* stream) {
  dlb::RaggedProblem pr{a, b, a_s, b_s, c, row_start, row_end, nullptr, 0, M_sum, N, K, G, expected_m, as_stride_m, as_stride_k, out_dtype,
                        false, nullptr, 0, 0, 0.f, static_cast<hipStream_t>(stream)};
  return dlb::run_ragged(pr);
}

int dlb_fp8_gemm_grouped_ragged_silu_quant(const void* a, const void* b, const float* a_s, const float* b_s, void* out_q, float* out_s,
                                           const int32_t* row_start, const int32_t* row_end, const int32_t* a_row_index,
                                           int64_t a_rows, int32_t expected_m, int64_t M_sum, int64_t N, int64_t K, int32_t G,
                                           int64_t as_stride_m, int64_t as_stride_k, int64_t os_stride_m, int64_t os_stride_k,
                                           float eps, void* stream) {
  dlb::RaggedProblem pr{a, b, a_s, b_s, out_q, row_start, row_end, a_row_index, a_rows, M_sum, N, K, G, expected_m, as_stride_m, as_stride_k,
                        DLB_OUT_BF16, true, out_s, os_stride_m, os_stride_k, eps, static_cast<hipStream_t>(stream)};
  return dlb::run_ragged(pr);
}

int dlb_expert_gate_up_ragged(const void* a, const void* b, const float* a_s, const float* b_s, void* out_q, float* out_s, const int32_t* row_start,
                              const int32_t* row_end, const int32_t* a_row_index, int64_t a_rows, int32_t expected_m, int64_t M_sum, int64_t N,
                              int64_t K, int32_t G, int64_t as_stride_m, int64_t as_stride_k, int64_t os_stride_m, int64_t os_stride_k, float eps,
                              void* workspace, size_t workspace_bytes, void* stream) {
  dlb::RaggedProblem pr{a, b, a_s, b_s, out_q, row_start, row_end, a_row_index, a_rows, M_sum, N, K, G, expected_m, as_stride_m, as_stride_k,
                        DLB_OUT_BF16, true, out_s, os_stride_m, os_stride_k, eps, static_cast<hipStream_t>(stream), workspace, workspace_bytes, true};
  return dlb::run_ragged(pr);
}

int dlb_expert_gate_up_masked(const void* a, const void* b, const float* a_s, const float* b_s, void* out_q, float* out_s, const int32_t* masked_m,
                              int32_t expected_m, int64_t M_max, int64_t N, int64_t K, int32_t G, int64_t as_stride_g, int64_t as_stride_m,
                              int64_t as_stride_k, int64_t os_stride_g, int64_t os_stride_m, int64_t os_stride_k, float eps, void* workspace,
                              size_t workspace_bytes, void* stream) {
  dlb::Problem pr{dlb::kMasked, a, b, a_s, b_s, out_q, masked_m, M_max, N, K, G, as_stride_g, as_stride_m, as_stride_k,
                  DLB_OUT_BF16, workspace, workspace_bytes, static_cast<hipStream_t>(stream)};
  pr.act = true;
  pr.mlp = true;
  pr.act_s = out_s;
  pr.act_s_sg = os_stride_g;
  pr.act_s_sm = os_stride_m;
  pr.act_s_sk = os_stride_k;
  pr.act_eps = eps;
  pr.hint_rows = expected_m;
  if (M_max > 0 && N > 0 && G > 0 && !out_s) return dlb::fail(DLB_ERR_NULL_POINTER, "out_s is NULL");
  return dlb::run(pr);
}

int dlb_expert_plan(int mode, int64_t rows, int64_t N, int64_t K, int32_t G, int32_t expected_m, int quantising, size_t workspace_bytes, int compute_units,
                    int* form) {
  dlb::clear_error();
  const int64_t lim = (1ll << 31) - 1024;
  if (rows < 0 || N < 0 || K < 0 || G < 0 || rows > lim || N > lim || K > lim || compute_units <= 0)
    return dlb::fail(DLB_ERR_BAD_SHAPE, "bad dimension (rows=%lld, N=%lld, K=%lld, G=%d)", (long long)rows, (long long)N, (long long)K, G);
  if (mode != dlb::kContiguous && mode != dlb::kMasked) return dlb::fail(DLB_ERR_BAD_SHAPE, "mode %d is not 1 (contiguous) or 2 (masked)", mode);
  if (!form) return DLB_OK;
  if (mode == dlb::kContiguous) {
    *form = dlb::expert_form(rows, N, K, G, expected_m, quantising != 0, workspace_bytes, compute_units);
  } else {
    const dlb::Resolved rs = dlb::resolve(dlb::kMasked, rows, N, K, G, dlb::ceil_div(K, dlb::kScaleBlock), 1, workspace_bytes > 0, workspace_bytes,
                                          compute_units, false, quantising != 0, expected_m, true, dlb::kMaxStreamSlices);
    const bool shape_ok = K > 0 && K % dlb::kScaleBlock == 0 && N % (2 * dlb::kScaleBlock) == 0 && N * K < (1ll << 32);
    *form = shape_ok && dlb::g_forced_variant < 0 && !dlb::steps_apart(rs, rows, N, G, expected_m, compute_units) ? 1 : 0;
  }
  return DLB_OK;
}

int dlb_fp8_quant_group(const void* x, int x_dtype, void* q, float* s, int64_t rows, int64_t K, int64_t group_size,
                        int64_t x_row_stride, int64_t s_stride_m, int64_t s_stride_k, float eps, void* stream) {
  using namespace dlb;
  g_err[0] = '\0';
  if (x_dtype < kInBf16 || x_dtype > kInF32) return fail(DLB_ERR_BAD_DTYPE, "x_dtype %d is not DLB_IN_BF16 / F16 / F32", x_dtype);
  if (rows < 0 || K < 0) return fail(DLB_ERR_BAD_SHAPE, "negative dimension (rows=%lld K=%lld)", (long long)rows, (long long)K);
  if (group_size <= 0) return fail(DLB_ERR_BAD_SHAPE, "group size %lld is not positive", (long long)group_size);
  if (K % group_size != 0)
    return fail(DLB_ERR_BAD_SHAPE, "K=%lld is not a multiple of the group size %lld", (long long)K, (long long)group_size);
  if (rows == 0 || K == 0) return DLB_OK;
  if (!x || !q || !s) return fail(DLB_ERR_NULL_POINTER, "x, q or s is NULL");
  const int64_t esz = x_dtype == kInF32 ? 4 : 2;
  if (x_row_stride < K) return fail(DLB_ERR_BAD_STRIDE, "x row stride %lld < K", (long long)x_row_stride);
  if (s_stride_m < 0 || s_stride_k < 0) return fail(DLB_ERR_BAD_STRIDE, "negative scale stride");
  if (misaligned(x, esz) || misaligned(s, 4)) return fail(DLB_ERR_ALIGNMENT, "x or s is not aligned to its element size");
  // the vector kernel: whole 16-byte loads and 8-byte stores per lane
  const bool vector_ok = group_size % 8 == 0 && group_size <= 512 && !misaligned(x, 16) && (x_row_stride * esz) % 16 == 0 && !misaligned(q, 8);
  if (group_size == kScaleBlock && !vector_ok) return fail(DLB_ERR_ALIGNMENT, "x rows must be 16-byte aligned, q 8-byte aligned");
  int lanes = 0;  // 0 = generic kernel
  if (vector_ok)
    for (lanes = 1; lanes * 8 < group_size; lanes *= 2) {
    }
  int dev = 0;
  const int cus = device_cu_count(&dev);
  if (cus < 0) return fail(DLB_ERR_LAUNCH, "hipGetDevice failed");
  QuantArgs qa{x, static_cast<uint8_t*>(q), s, rows, K / group_size, group_size, x_row_stride, s_stride_m, s_stride_k, eps};
  const int64_t groups = rows * (K / group_size);
  const int64_t per_block = lanes > 0 ? 4 * (64 / lanes) : 4;  // 4 waves x groups per wave and step
  int64_t blocks = ceil_div(groups, per_block);
  const int64_t cap = static_cast<int64_t>(cus) * 16;
  if (blocks > cap) blocks = cap;
  hipStream_t st = static_cast<hipStream_t>(stream);
  if (x_dtype == kInBf16)
    launch_quant_group<kInBf16>(qa, lanes, static_cast<unsigned>(blocks), st);
  else if (x_dtype == kInF16)
    launch_quant_group<kInF16>(qa, lanes, static_cast<unsigned>(blocks), st);
  else
    launch_quant_group<kInF32>(qa, lanes, static_cast<unsigned>(blocks), st);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e));
  return DLB_OK;
}

int dlb_fp8_quant_1x128(const void* x, int x_dtype, void* q, float* s, int64_t rows, int64_t K, int64_t x_row_stride,
                        int64_t s_stride_m, int64_t s_stride_k, float eps, void* stream) {
  return dlb_fp8_quant_group(x, x_dtype, q, s, rows, K, dlb::kScaleBlock, x_row_stride, s_stride_m, s_stride_k, eps, stream);
}

int dlb_fp8_quant_128x128(const void* w, int w_dtype, void* q, float* s, int64_t G, int64_t N, int64_t K,
                          int64_t w_row_stride, float eps, void* stream) {
  using namespace dlb;
  g_err[0] = '\0';
  if (w_dtype < kInBf16 || w_dtype > kInF32) return fail(DLB_ERR_BAD_DTYPE, "w_dtype %d is not DLB_IN_BF16 / F16 / F32", w_dtype);
  if (G < 0 || N < 0 || K < 0)
    return fail(DLB_ERR_BAD_SHAPE, "negative dimension (G=%lld N=%lld K=%lld)", (long long)G, (long long)N, (long long)K);
  if (K % 8 != 0) return fail(DLB_ERR_BAD_SHAPE, "K=%lld is not a multiple of 8", (long long)K);
  if (G == 0 || N == 0 || K == 0) return DLB_OK;
  if (!w || !q || !s) return fail(DLB_ERR_NULL_POINTER, "w, q or s is NULL");
  const int64_t esz = w_dtype == kInF32 ? 4 : 2;
  if (w_row_stride < K) return fail(DLB_ERR_BAD_STRIDE, "w row stride %lld < K", (long long)w_row_stride);
  if (misaligned(w, 16) || (w_row_stride * esz) % 16 != 0 || misaligned(q, 8) || misaligned(s, 4))
    return fail(DLB_ERR_ALIGNMENT, "w rows must be 16-byte aligned, q 8-byte aligned");
  const int64_t nbn = ceil_div(N, kScaleBlock), nbk = ceil_div(K, kScaleBlock);
  const int64_t blocks = G * nbn * nbk;
  if (blocks >= (1ll << 31) || nbn >= (1ll << 30) || nbk >= (1ll << 30)) return fail(DLB_ERR_BAD_SHAPE, "too many blocks");
  BlockQuantArgs a{w, static_cast<uint8_t*>(q), s, N, K, w_row_stride, static_cast<int>(nbn), static_cast<int>(nbk), eps};
  hipStream_t st = static_cast<hipStream_t>(stream);
  const dim3 grid(static_cast<unsigned>(blocks)), block(256);
  if (w_dtype == kInBf16)
    hipLaunchKernelGGL(fp8_quant_128x128_kernel<kInBf16>, grid, block, 0, st, a);
  else if (w_dtype == kInF16)
    hipLaunchKernelGGL(fp8_quant_128x128_kernel<kInF16>, grid, block, 0, st, a);
  else
    hipLaunchKernelGGL(fp8_quant_128x128_kernel<kInF32>, grid, block, 0, st, a);
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "kernel launch failed: %s", hipGetErrorString(e));
  return DLB_OK;
}

int dlb_fp8_gemm_plan(int mode, int64_t rows, int64_t N, int64_t K, size_t workspace_bytes, int compute_units, int* variant,
                      int* k_slices, int* decode_columns, int64_t* narrow_from) {
  dlb::clear_error();
  if (mode < dlb::kDense || mode > dlb::kMasked) return dlb::fail(DLB_ERR_BAD_SHAPE, "mode %d is not 0 (dense), 1 (contiguous) or 2 (masked)", mode);
  if (rows < 0 || N < 0 || K < 0) return dlb::fail(DLB_ERR_BAD_SHAPE, "negative dimension (rows=%lld, N=%lld, K=%lld)", (long long)rows, (long long)N, (long long)K);
  const int64_t lim = (1ll << 31) - 1024;
  if (rows > lim || N > lim || K > lim) return dlb::fail(DLB_ERR_BAD_SHAPE, "dimension beyond 2^31");
  if (compute_units <= 0) return dlb::fail(DLB_ERR_BAD_SHAPE, "compute_units must be positive");
  // row-major activation scales, as the dense Python entry point hands them over
  const dlb::Resolved rs = dlb::resolve(mode, rows, N, K, mode == dlb::kDense ? 1 : 32, dlb::ceil_div(K, dlb::kScaleBlock), 1,
                                        workspace_bytes > 0, workspace_bytes, compute_units, false, false, -1, false);
  if (variant) *variant = rs.pl.variant;
  if (k_slices) *k_slices = rs.splitk;
  if (decode_columns) *decode_columns = dlb::is_skinny(rs.pl.variant) ? rs.pl.sk_bn : 0;
  if (narrow_from) *narrow_from = rs.n_split;
  return DLB_OK;
}

int dlb_fp8_gemm_plan_wave_k(int64_t M, int64_t N, int64_t K, size_t workspace_bytes, int compute_units, int* tile_rows, int* tile_columns,
                             int* waves) {
  dlb::clear_error();
  const int64_t lim = (1ll << 31) - 1024;
  if (M < 0 || N < 0 || K < 0 || M > lim || N > lim || K > lim || compute_units <= 0)
    return dlb::fail(DLB_ERR_BAD_SHAPE, "bad dimension (M=%lld, N=%lld, K=%lld)", (long long)M, (long long)N, (long long)K);
  const dlb::Resolved rs = dlb::resolve(dlb::kDense, M, N, K, 1, dlb::ceil_div(K, dlb::kScaleBlock), 1, workspace_bytes > 0, workspace_bytes,
                                        compute_units);
  const bool on = rs.wavek != dlb::kWaveKNone;
  if (tile_rows) *tile_rows = on ? 32 * dlb::kWaveKDims[rs.wavek].mf : 0;
  if (tile_columns) *tile_columns = on ? 32 * dlb::kWaveKDims[rs.wavek].nf : 0;
  if (waves) *waves = on ? dlb::kWaveKDims[rs.wavek].waves : 0;
  return DLB_OK;
}

int dlb_fp8_gemm_plan_grouped(int mode, int64_t rows, int64_t N, int64_t K, int32_t G, int32_t expected_m, size_t workspace_bytes,
                              int compute_units, int* variant, int* tile_lists) {
  dlb::clear_error();
  if (mode != dlb::kContiguous && mode != dlb::kMasked) return dlb::fail(DLB_ERR_BAD_SHAPE, "mode %d is not 1 (contiguous) or 2 (masked)", mode);
  if (rows < 0 || N < 0 || K < 0 || G < 0) return dlb::fail(DLB_ERR_BAD_SHAPE, "negative dimension (rows=%lld, N=%lld, K=%lld, G=%d)", (long long)rows, (long long)N, (long long)K, G);
  const int64_t lim = (1ll << 31) - 1024;
  if (rows > lim || N > lim || K > lim) return dlb::fail(DLB_ERR_BAD_SHAPE, "dimension beyond 2^31");
  if (compute_units <= 0) return dlb::fail(DLB_ERR_BAD_SHAPE, "compute_units must be positive");
  const dlb::Resolved rs = dlb::resolve(mode, rows, N, K, G, dlb::ceil_div(K, dlb::kScaleBlock), 1, workspace_bytes > 0, workspace_bytes,
                                        compute_units, false, false, mode == dlb::kMasked ? expected_m : -1);
  if (variant) *variant = rs.pl.variant;
  if (tile_lists) *tile_lists = rs.tile_list ? 1 : 0;
  return DLB_OK;
}

int dlb_fp8_gemm_plan_stream_launch(int mode, int64_t rows, int64_t N, int64_t K, int32_t G, int32_t expected_m, int quantising, int mlp,
                                    size_t workspace_bytes, int compute_units, int* tile_rows, int* tile_columns, int* ahead, int* slices) {
  dlb::clear_error();
  const int64_t lim = (1ll << 31) - 1024;
  if (rows < 0 || N < 0 || K < 0 || G < 0 || rows > lim || N > lim || K > lim || compute_units <= 0)
    return dlb::fail(DLB_ERR_BAD_SHAPE, "bad dimension (rows=%lld, N=%lld, K=%lld, G=%d)", (long long)rows, (long long)N, (long long)K, G);
  if (mode != dlb::kContiguous && mode != dlb::kMasked) return dlb::fail(DLB_ERR_BAD_SHAPE, "mode %d is not 1 (contiguous) or 2 (masked)", mode);
  const bool act = quantising != 0;
  dlb::StreamPlan sp;
  if (mode == dlb::kContiguous) {
    sp = dlb::ragged_stream(rows, N, K, G, expected_m, act, mlp != 0, workspace_bytes, compute_units);
  } else if (!act || (N % (2 * dlb::kScaleBlock) == 0 && N * K < (1ll << 32))) {
    sp = dlb::resolve(dlb::kMasked, rows, N, K, G, dlb::ceil_div(K, dlb::kScaleBlock), 1, workspace_bytes > 0, workspace_bytes, compute_units, false, act,
                      expected_m, true, mlp != 0 ? dlb::kMaxStreamSlices : 1)
             .stream;
  }
  const bool on = sp.shape != dlb::kStreamNone;
  if (tile_rows) *tile_rows = on ? dlb::kStreamDims[sp.shape].bm : 0;
  if (tile_columns) *tile_columns = on ? dlb::kStreamDims[sp.shape].bn : 0;
  if (ahead) *ahead = on && sp.ahead ? 1 : 0;
  if (slices) *slices = on ? sp.slices : 0;
  return DLB_OK;
}

int dlb_fp8_gemm_plan_stream(int64_t rows, int64_t N, int64_t K, int32_t G, int32_t expected_m, int quantising, int compute_units,
                             int* tile_rows, int* tile_columns, int* ahead) {
  return dlb_fp8_gemm_plan_stream_launch(dlb::kMasked, rows, N, K, G, expected_m, quantising, 0, 0, compute_units, tile_rows, tile_columns, ahead, nullptr);
}

int dlb_fp8_gemm_force_variant(int variant) {
  if (variant >= dlb::kVarCount) return dlb::fail(DLB_ERR_BAD_SHAPE, "unknown kernel variant %d", variant);
  dlb::g_forced_variant = variant < 0 ? -1 : variant;
  return DLB_OK;
}

int dlb_fp8_gemm_tune(int knob, int value) {
  if (knob < 0 || knob >= dlb::kKnobCount) return dlb::fail(DLB_ERR_BAD_SHAPE, "unknown tuning knob %d", knob);
  if (value < 0 || value > 1024) return dlb::fail(DLB_ERR_BAD_SHAPE, "tuning value %d outside [0, 1024]", value);
  dlb::g_knob[knob] = value;
  return DLB_OK;
}

const char* dlb_fp8_gemm_variant_name(int variant) {
  if (variant < 0 || variant >= dlb::kVarCount) return nullptr;
  return dlb::kVariantNames[variant];
}

// declared in include/dlblas_fp8_moe.h; lives here next to the kernel it shares with the GEMM's own pre-pass
int dlb_scale_relayout(const float* src, float* dst, int64_t rows, int64_t kblocks, int64_t rows_pad,
                       int64_t src_stride_m, int64_t src_stride_k, void* stream) {
  using namespace dlb;
  clear_error();
  if (rows < 0 || kblocks < 0 || rows_pad < rows)
    return fail(DLB_ERR_BAD_SHAPE, "bad dimensions (rows=%lld kblocks=%lld rows_pad=%lld)", (long long)rows, (long long)kblocks,
                (long long)rows_pad);
  if (rows_pad == 0 || kblocks == 0) return DLB_OK;
  if (!dst || (rows > 0 && !src)) return fail(DLB_ERR_NULL_POINTER, "src or dst is NULL");
  if (rows_pad >= (1ll << 31) || kblocks >= (1ll << 31) || ceil_div(kblocks, 32) > 65535)
    return fail(DLB_ERR_BAD_SHAPE, "dimensions beyond the supported range");
  const dim3 grid(static_cast<unsigned>(ceil_div(rows_pad, 32)), static_cast<unsigned>(ceil_div(kblocks, 32)), 1);
  hipLaunchKernelGGL(fp8_scale_transpose_kernel, grid, dim3(256), 0, static_cast<hipStream_t>(stream), src, dst,
                     static_cast<int>(rows), static_cast<int>(kblocks), static_cast<int>(rows_pad), static_cast<int64_t>(0),
                     src_stride_m, src_stride_k, static_cast<const int32_t*>(nullptr));
  const hipError_t e = hipGetLastError();
  if (e != hipSuccess) return fail(DLB_ERR_LAUNCH, "scale_relayout launch failed: %s", hipGetErrorString(e));
  return DLB_OK;
}

}  // extern "C"
