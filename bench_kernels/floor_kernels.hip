// Bench-only kernels (not part of the library): what this GPU allows the GEMM kernels' instruction mix and access
// patterns when everything else is taken away.  bench.py times them (--decode-floor, --ceilings):
//   floor_empty  a kernel with the decode kernel's grid and block that returns at once: the per-launch cost of the
//                queue (dependent launches on one stream)
//   floor_read   every byte of the weight matrix read once with 16-byte loads, nothing else: launch cost + the time the
//                memory system needs to deliver the bytes to 256 workgroups
//   floor_mfma   the prefill kernels' arithmetic and nothing else, two waves per SIMD: MFMAs on a zero accumulator, scale FMAs two MFMAs
//                behind.  Form 1: the kernels' 16 x 16 x 128, 32 of them and 128 FMAs per K step of a 64 x 128 wave tile, from registers;
//                form 2: the same with every fragment read from LDS, at the kernels' distance ahead of its use; form 0: the same
//                products as pairs of 32 x 32 x 64 from registers.  The operands come from the caller, so that the same loop runs on
//                constant and on random e4m3 codes
//   floor_panel_stream  one workgroup per CU streams 256-row panels of a row-major byte matrix through the LDS DMA path
//                (global_load_lds_dwordx4, 8 rows x 128 bytes per wave instruction, K step by K step, S steps in
//                flight) and does nothing with them: the rate at which a CU can pull a weight tile's rows from HBM
//   floor_l2_stream  one workgroup per CU pulls the SAME 512 rows of a row-major byte matrix, 128 bytes per row and K
//                step (the 64 KB a 256 x 256 GEMM tile needs per K step), so that after the first touch every request
//                hits the L2: what the path from the L2 into a CU delivers, through the LDS DMA (S steps in flight) or
//                through 16-byte register loads
#include <hip/hip_runtime.h>
#include <stdint.h>

typedef int v4i __attribute__((ext_vector_type(4)));
typedef int v8i __attribute__((ext_vector_type(8)));
typedef float v4f __attribute__((ext_vector_type(4)));
typedef float v16f __attribute__((ext_vector_type(16)));
typedef __attribute__((address_space(3))) void* lds_ptr_t;
typedef const __attribute__((address_space(1))) void* global_ptr_t;

__global__ void __launch_bounds__(512) floor_empty_kernel(int* sink) {
  if (sink == reinterpret_cast<int*>(1)) *sink = 0;  // never true: keeps the argument alive
}

// grid-stride over 16-byte words, U loads in flight per thread; the xor of everything read is stored only if it equals
// a value it cannot take, so the loads stay and nothing is written
template <int U>
__global__ void __launch_bounds__(512) floor_read_kernel(const v4i* src, int64_t words, int* sink) {
  v4i acc = {0, 0, 0, 0};
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i + (U - 1) * stride < words; i += U * stride) {
    v4i v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(src + i + u * stride);
#pragma unroll
    for (int u = 0; u < U; ++u) acc ^= v[u];
  }
  for (; i < words; i += stride) acc ^= __builtin_nontemporal_load(src + i);
  if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x5a5a5a5a && sink == reinterpret_cast<int*>(1)) *sink = acc.x;
}

// The same reads, then what any GEMM of that shape also has to do at its end: one exchange between the waves of a
// workgroup through LDS (a barrier) and the store of the workgroup's share of `out_bytes` of output.
template <int U>
__global__ void __launch_bounds__(512) floor_read_store_kernel(const v4i* src, int64_t words, int* out, int64_t out_bytes) {
  __shared__ int xch[512];
  v4i acc = {0, 0, 0, 0};
  const int64_t stride = static_cast<int64_t>(gridDim.x) * blockDim.x;
  int64_t i = static_cast<int64_t>(blockIdx.x) * blockDim.x + threadIdx.x;
  for (; i + (U - 1) * stride < words; i += U * stride) {
    v4i v[U];
#pragma unroll
    for (int u = 0; u < U; ++u) v[u] = __builtin_nontemporal_load(src + i + u * stride);
#pragma unroll
    for (int u = 0; u < U; ++u) acc ^= v[u];
  }
  for (; i < words; i += stride) acc ^= __builtin_nontemporal_load(src + i);
  xch[threadIdx.x] = acc.x ^ acc.y ^ acc.z ^ acc.w;
  __syncthreads();
  const int mixed = xch[threadIdx.x] ^ xch[(threadIdx.x + 64) & 511] ^ xch[(threadIdx.x + 192) & 511];
  const int64_t per_wg = out_bytes / 4 / gridDim.x;  // dwords of output per workgroup
  for (int64_t t = threadIdx.x; t < per_wg; t += 512) out[static_cast<int64_t>(blockIdx.x) * per_wg + t] = mixed;
}

// in: 8 x 64 x 32 bytes of e4m3 codes
__global__ void __launch_bounds__(512) floor_mfma_pairs_kernel(const v8i* in, float* out, int iters, float scale) {
  const int lane = threadIdx.x & 63;
  v8i a[4], b[2];
  for (int i = 0; i < 4; ++i) a[i] = in[lane + 64 * i];
  for (int i = 0; i < 2; ++i) b[i] = in[lane + 64 * (4 + i)];
  v16f acc[4], part[2];
  for (int j = 0; j < 16; ++j) acc[0][j] = acc[1][j] = acc[2][j] = acc[3][j] = part[0][j] = part[1][j] = 0.0f;
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int t = 0; t < 8; ++t) {
      if (t % 4 == 0) asm volatile("" : "+v"(a[0][0]), "+v"(a[1][0]), "+v"(a[2][0]), "+v"(a[3][0]));  // no four pairs are copies of others
      __builtin_amdgcn_sched_barrier(0);
      v16f z;
      for (int j = 0; j < 16; ++j) z[j] = 0.0f;
      z = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[t & 3], b[0], z, 0, 0, 0, 0, 0, 0);
      part[t & 1] = __builtin_amdgcn_mfma_scale_f32_32x32x64_f8f6f4(a[(t + 1) & 3], b[1], z, 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      acc[(t + 3) & 3] += part[(t + 1) & 1] * scale;  // the scale FMAs of the previous pair
    }
  }
  float r = 0.0f;
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 16; ++j) r += acc[i][j];
  out[blockIdx.x * 512 + threadIdx.x] = r;
}

// in: as above.  LDS: a 64 KB copy of it, read row by row as 128-byte rows of K; the reads are ordinary loads, whose waits the compiler places.
template <bool LDS>
__global__ void __launch_bounds__(512) floor_mfma_kernel(const v8i* in, float* out, int iters, float scale) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  if (LDS) {
    for (int i = threadIdx.x; i < 65536 / 16; i += 512) reinterpret_cast<v4i*>(lds)[i] = reinterpret_cast<const v4i*>(in)[i % 1024];
    __syncthreads();
  }
  // fragment f of a stage: rows f / 2 * 32 + f % 2 * 4 + ..., chunk pattern without bank conflicts, as in the ring kernels
  const int row = ((lane & 15) >> 2) * 8 + (lane & 3), q = lane >> 4;
  const int at = row * 128 + (((((q & 1) * 2 + (q >> 1)) ^ ((row & 2) | ((row >> 3) & 1) | ((row >> 2) & 4))) & 7) << 4);
  auto read = [&](int stage, int f) {  // stage: 0 or 1, 32 KB each; held fragments are 0 .. 3, streamed ones 4 .. 11
    const int base = stage * 32768 + (wave & 3) * 1024 + f / 2 * 4096 + f % 2 * 512 + at;  // ends at 60416 at most
    const v4i lo = *reinterpret_cast<const v4i*>(lds + base), hi = *reinterpret_cast<const v4i*>(lds + (base ^ 64));
    return v8i{lo.x, lo.y, lo.z, lo.w, hi.x, hi.y, hi.z, hi.w};
  };
  v8i held[4], strm[4];
  for (int i = 0; i < 4; ++i) held[i] = in[lane + 64 * i], strm[i] = in[lane + 64 * (4 + i)];
  v4f acc[4][8], part[4];
  for (int i = 0; i < 4; ++i) {
    part[i] = v4f{0.0f, 0.0f, 0.0f, 0.0f};
    for (int j = 0; j < 8; ++j) acc[i][j] = part[i];
  }
  for (int it = 0; it < iters; ++it) {
#pragma unroll
    for (int s = 0; s < 32; ++s) {
      const int n = s / 4, m = s % 4, behind = (s + 30) % 32;
      if (!LDS && s % 16 == 0) asm volatile("" : "+v"(held[0][0]), "+v"(held[1][0]), "+v"(held[2][0]), "+v"(held[3][0]));  // no 16 products are copies of others
      __builtin_amdgcn_sched_barrier(0);
      part[s % 4] = __builtin_amdgcn_mfma_scale_f32_16x16x128_f8f6f4(strm[n % 4], held[m], v4f{0.0f, 0.0f, 0.0f, 0.0f}, 0, 0, 0, 0, 0, 0);
      __builtin_amdgcn_sched_barrier(0);
      if (LDS && m == 0) strm[(n + 3) % 4] = read((it + (n + 3) / 8) & 1, 4 + (n + 3) % 8);
      if (LDS && n == 7) held[m] = read((it + 1) & 1, m);
      __builtin_amdgcn_sched_barrier(0);
      acc[behind % 4][behind / 4] += part[behind % 4] * scale;
      __builtin_amdgcn_sched_barrier(0);
    }
  }
  float r = 0.0f;
  for (int i = 0; i < 4; ++i)
    for (int j = 0; j < 8; ++j) r += acc[i][j].x + acc[i][j].y + acc[i][j].z + acc[i][j].w;
  out[blockIdx.x * 512 + threadIdx.x] = r;
}

// S = K steps a wave keeps in flight.  Matrix [panels * 256][row_bytes]; workgroup b takes panels b, b + grid, ...
// POLICY = cache-policy operand of the loads of src (0, or 2 = the non-temporal bit); the shared panel always uses 0
template <int S, int POLICY>
__global__ void __launch_bounds__(512) floor_panel_stream_kernel(const char* src, int panels, int64_t row_bytes, const char* hot,
                                                                 int hot_panels) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ksteps = static_cast<int>(row_bytes / 128);
  for (int p = blockIdx.x; p < panels; p += gridDim.x) {
    // lane -> (row of the wave's 32, 16-byte chunk of the row's 128-byte line)
    const char* base = src + (static_cast<int64_t>(p) * 256 + wave * 32 + (lane >> 3)) * row_bytes + (lane & 7) * 16;
    for (int k = 0; k < ksteps; ++k) {
#pragma unroll
      for (int u = 0; u < 4; ++u)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(base + static_cast<int64_t>(u) * 8 * row_bytes + k * 128),
                                         (lds_ptr_t)(lds + ((k % S) * 32 + wave * 4 + u) * 1024), 16, 0, POLICY);
      if (hot != nullptr) {
        // a second 256-row panel per K step that many workgroups share (the activation strip of a GEMM tile: L2 hits)
        const char* hbase = hot + (static_cast<int64_t>((p / 16) % hot_panels) * 256 + wave * 32 + (lane >> 3)) * row_bytes + (lane & 7) * 16;
#pragma unroll
        for (int u = 0; u < 4; ++u)
          __builtin_amdgcn_global_load_lds((global_ptr_t)(hbase + static_cast<int64_t>(u) * 8 * row_bytes + k * 128),
                                           (lds_ptr_t)(lds + ((k % S) * 32 + wave * 4 + u) * 1024), 16, 0, 0);
        if (S == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
        if (S == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
        if (S == 4) asm volatile("s_waitcnt vmcnt(24)" ::: "memory");
        continue;
      }
      if (S == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (S == 2) asm volatile("s_waitcnt vmcnt(4)" ::: "memory");
      if (S == 4) asm volatile("s_waitcnt vmcnt(12)" ::: "memory");
    }
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
}

// MODE 0: global_load_lds_dwordx4 into a ring of S stages of 64 KB; MODE 1: global_load_dwordx4 into registers, the
// loads of S K steps (8 per wave and step) in flight.  Workgroup b starts its walk over K at step 7 b (mod ksteps).
template <int MODE, int S>
__global__ void __launch_bounds__(512) floor_l2_stream_kernel(const char* src, int64_t row_bytes, int iters, int* sink) {
  extern __shared__ __attribute__((aligned(16))) char lds[];
  const int lane = threadIdx.x & 63, wave = threadIdx.x >> 6;
  const int ksteps = static_cast<int>(row_bytes / 128);
  const char* base = src + (static_cast<int64_t>(wave) * 64 + (lane >> 3)) * row_bytes + (lane & 7) * 16;
  int k = static_cast<int>((blockIdx.x * 7u) % static_cast<unsigned>(ksteps));
  v4i acc = {0, 0, 0, 0};
  for (int it = 0; it < iters; ++it) {
    if (MODE == 0) {
#pragma unroll
      for (int u = 0; u < 8; ++u)
        __builtin_amdgcn_global_load_lds((global_ptr_t)(base + static_cast<int64_t>(u) * 8 * row_bytes + k * 128),
                                         (lds_ptr_t)(lds + ((it % S) * 64 + wave * 8 + u) * 1024), 16, 0, 0);
      if (S == 1) asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
      if (S == 2) asm volatile("s_waitcnt vmcnt(8)" ::: "memory");
    } else {
      v4i v[S][8];
#pragma unroll
      for (int s2 = 0; s2 < S; ++s2) {
#pragma unroll
        for (int u = 0; u < 8; ++u)
          v[s2][u] = *reinterpret_cast<const v4i*>(base + static_cast<int64_t>(u) * 8 * row_bytes + k * 128);
        k = k + 1 == ksteps ? 0 : k + 1;
      }
#pragma unroll
      for (int s2 = 0; s2 < S; ++s2)
#pragma unroll
        for (int u = 0; u < 8; ++u) acc ^= v[s2][u];
      it += S - 1;
      continue;
    }
    k = k + 1 == ksteps ? 0 : k + 1;
  }
  asm volatile("s_waitcnt vmcnt(0)" ::: "memory");
  if ((acc.x ^ acc.y ^ acc.z ^ acc.w) == 0x5a5a5a5a && sink == reinterpret_cast<int*>(1)) *sink = acc.x;
}

extern "C" {

// src: [512][row_bytes] bytes; K steps of 64 KB per workgroup = iters; mode 0 = LDS DMA, 1 = register loads; depth = K
// steps in flight (1 or 2)
int floor_l2_stream(const void* src, int64_t row_bytes, int workgroups, int iters, int mode, int depth, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const char* p = static_cast<const char*>(src);
  if (row_bytes <= 0 || row_bytes % 128 != 0) return -1;
  auto launch = [&](auto kernel, int lds_bytes) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 131072) != hipSuccess) return;
    hipLaunchKernelGGL(kernel, dim3(workgroups), dim3(512), lds_bytes, st, p, row_bytes, iters, nullptr);
  };
  if (mode == 0 && depth >= 2) launch(floor_l2_stream_kernel<0, 2>, 131072);
  if (mode == 0 && depth < 2) launch(floor_l2_stream_kernel<0, 1>, 65536);
  if (mode != 0 && depth >= 2) launch(floor_l2_stream_kernel<1, 2>, 0);
  if (mode != 0 && depth < 2) launch(floor_l2_stream_kernel<1, 1>, 0);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int floor_empty(int workgroups, void* stream) {
  hipLaunchKernelGGL(floor_empty_kernel, dim3(workgroups), dim3(512), 0, static_cast<hipStream_t>(stream), nullptr);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// loads_in_flight: 16-byte loads each thread issues before it uses the first (2, 4 or 8)
int floor_read(const void* src, int64_t bytes, int workgroups, int loads_in_flight, void* stream) {
  const dim3 grid(workgroups), block(512);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const v4i* p = static_cast<const v4i*>(src);
  if (loads_in_flight >= 8)
    hipLaunchKernelGGL(floor_read_kernel<8>, grid, block, 0, st, p, bytes / 16, nullptr);
  else if (loads_in_flight >= 4)
    hipLaunchKernelGGL(floor_read_kernel<4>, grid, block, 0, st, p, bytes / 16, nullptr);
  else
    hipLaunchKernelGGL(floor_read_kernel<2>, grid, block, 0, st, p, bytes / 16, nullptr);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int floor_read_store(const void* src, int64_t bytes, int workgroups, int loads_in_flight, void* out, int64_t out_bytes, void* stream) {
  const dim3 grid(workgroups), block(512);
  hipStream_t st = static_cast<hipStream_t>(stream);
  const v4i* p = static_cast<const v4i*>(src);
  int* o = static_cast<int*>(out);
  if (loads_in_flight >= 8)
    hipLaunchKernelGGL(floor_read_store_kernel<8>, grid, block, 0, st, p, bytes / 16, o, out_bytes);
  else if (loads_in_flight >= 4)
    hipLaunchKernelGGL(floor_read_store_kernel<4>, grid, block, 0, st, p, bytes / 16, o, out_bytes);
  else
    hipLaunchKernelGGL(floor_read_store_kernel<2>, grid, block, 0, st, p, bytes / 16, o, out_bytes);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// operands: 16384 bytes of e4m3 codes on the device; out: workgroups * 512 floats; form 0, 1 or 2 (above).  FLOP per launch =
// workgroups * 8 waves * iters * 2097152 in every form.
int floor_mfma(const void* operands, float* out, int workgroups, int iters, int form, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const v8i* in = static_cast<const v8i*>(operands);
  if (form == 0) {
    hipLaunchKernelGGL(floor_mfma_pairs_kernel, dim3(workgroups), dim3(512), 0, st, in, out, iters, 1.5f);
  } else if (form == 1) {
    hipLaunchKernelGGL(floor_mfma_kernel<false>, dim3(workgroups), dim3(512), 0, st, in, out, iters, 1.5f);
  } else {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(floor_mfma_kernel<true>), hipFuncAttributeMaxDynamicSharedMemorySize, 65536) != hipSuccess) return -1;
    hipLaunchKernelGGL(floor_mfma_kernel<true>, dim3(workgroups), dim3(512), 65536, st, in, out, iters, 1.5f);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// src: [panels * 256][row_bytes] bytes, row_bytes a multiple of 128; steps_in_flight 1, 2 or 4; non_temporal: the loads
// of src carry the non-temporal bit; hot: nullptr, or
// [hot_panels * 256][row_bytes] bytes of which every workgroup also pulls one panel per panel of src (16 consecutive
// panels of src share one)
int floor_panel_stream(const void* src, int panels, int64_t row_bytes, int workgroups, int steps_in_flight, const void* hot,
                       int hot_panels, int non_temporal, void* stream) {
  hipStream_t st = static_cast<hipStream_t>(stream);
  const char* p = static_cast<const char*>(src);
  const char* h = static_cast<const char*>(hot);
  if (hot != nullptr && hot_panels <= 0) return -1;
  if (row_bytes <= 0 || row_bytes % 128 != 0 || panels <= 0) return -1;
  const dim3 grid(workgroups), block(512);
  const int s = steps_in_flight >= 4 ? 4 : (steps_in_flight >= 2 ? 2 : 1);
  auto launch = [&](auto kernel) {
    if (hipFuncSetAttribute(reinterpret_cast<const void*>(kernel), hipFuncAttributeMaxDynamicSharedMemorySize, 131072) != hipSuccess) return;
    hipLaunchKernelGGL(kernel, grid, block, s * 32768, st, p, panels, row_bytes, h, hot_panels);
  };
  if (non_temporal) {
    if (s == 4) launch(floor_panel_stream_kernel<4, 2>);
    if (s == 2) launch(floor_panel_stream_kernel<2, 2>);
    if (s == 1) launch(floor_panel_stream_kernel<1, 2>);
  } else {
    if (s == 4) launch(floor_panel_stream_kernel<4, 0>);
    if (s == 2) launch(floor_panel_stream_kernel<2, 0>);
    if (s == 1) launch(floor_panel_stream_kernel<1, 0>);
  }
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // extern "C"
