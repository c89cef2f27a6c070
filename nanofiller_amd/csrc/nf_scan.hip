// nf_scan.hip - exclusive prefix sum over u32 arrays and fill kernels.
//
// Replaces the thrust::inclusive_scan / exclusive_scan calls of the
// reference (src/get_contact_arrays.cu:101, src/conductivity.cu:495,
// src/adjacency_graph.cu:79) and its in-block work-efficient scan
// (inc/sort.h:103-154).  Tiles of 2048 elements, 256 threads x 8
// items.  Two passes (tile sums; tile scan, each workgroup adding up the sums
// before its own) for up to 2048 tiles, three (the tile sums scanned between
// them) beyond, and for arrays of at most 16384 one pass of one workgroup;
// fixed launch shape for a given n, so the passes can be captured in a HIP
// graph.
#include "nf_internal.h"

namespace nf {

constexpr int SCAN_THREADS = 256;
constexpr int SCAN_ITEMS = 8;
constexpr int SCAN_TILE = SCAN_THREADS * SCAN_ITEMS;
constexpr uint32_t SUMS_MAX = 2048;

__device__ __forceinline__ uint32_t wave_incl_scan(uint32_t v) {
  const int lane = threadIdx.x & (WAVE - 1);
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const uint32_t t = __shfl_up(v, o, WAVE);
    v += (lane >= o) ? t : 0u;
  }
  return v;
}

// Exclusive scan of one value per thread over a 256-thread block.
__device__ __forceinline__ uint32_t block_excl_scan(uint32_t v, uint32_t* sm, uint32_t* total) {
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = threadIdx.x / WAVE;
  const uint32_t inc = wave_incl_scan(v);
  if (lane == WAVE - 1) sm[wv] = inc;
  __syncthreads();
  uint32_t off = 0, tot = 0;
#pragma unroll
  for (int w = 0; w < SCAN_THREADS / WAVE; ++w) {
    const uint32_t s = sm[w];
    if (w < wv) off += s;
    tot += s;
  }
  __syncthreads();
  *total = tot;
  return off + inc - v;
}

// The thread's eight elements, zero past the end.
__device__ __forceinline__ void scan_load(const uint32_t* __restrict__ in, uint64_t base, uint64_t n, bool wide,
                                          uint32_t v[SCAN_ITEMS]) {
  if (wide && base + SCAN_ITEMS <= n) {
    const uint4 a = *(const uint4*)(in + base), b = *(const uint4*)(in + base + 4);
    v[0] = a.x;
    v[1] = a.y;
    v[2] = a.z;
    v[3] = a.w;
    v[4] = b.x;
    v[5] = b.y;
    v[6] = b.z;
    v[7] = b.w;
    return;
  }
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint64_t i = base + k;
    const uint32_t x = in[i < n ? i : n - 1];  // clamped load, masked below
    v[k] = i < n ? x : 0u;
  }
}

// Elements that count: all, or as many as the device says (limit).
__device__ __forceinline__ uint64_t scan_length(uint64_t n, const uint32_t* limit) {
  return limit != nullptr && *limit < n ? *limit : n;
}

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_tiles(const uint32_t* __restrict__ in, uint64_t n,
                                                             const uint32_t* limit, bool wide,
                                                             uint32_t* __restrict__ sums) {
  __shared__ uint32_t sm[SCAN_THREADS / WAVE];
  n = scan_length(n, limit);
  if ((uint64_t)blockIdx.x * SCAN_TILE >= n) return;
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS], s = 0;
  scan_load(in, base, n, wide, v);
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) s += v[k];
  uint32_t tot;
  block_excl_scan(s, sm, &tot);
  if (threadIdx.x == 0) sums[blockIdx.x] = tot;
}

__global__ void __launch_bounds__(SCAN_THREADS) k_scan_sums(uint32_t* __restrict__ sums,
                                                            uint32_t nt, uint32_t* __restrict__ out,
                                                            uint64_t n, const uint32_t* limit) {
  n = scan_length(n, limit);
  nt = min(nt, (uint32_t)((n + SCAN_TILE - 1) / SCAN_TILE));
  __shared__ uint32_t sm[SCAN_THREADS / WAVE];
  __shared__ uint32_t dummy[SCAN_THREADS];
  uint32_t carry = 0;
  for (uint32_t b = 0; b < nt; b += SCAN_THREADS) {
    const uint32_t i = b + threadIdx.x;
    const uint32_t v = sums[i < nt ? i : nt - 1];
    uint32_t tot;
    const uint32_t ex = block_excl_scan(i < nt ? v : 0u, sm, &tot);
    // branch-free store: out-of-range threads write a private LDS slot
    uint32_t* dst = i < nt ? &sums[i] : &dummy[threadIdx.x];
    *dst = carry + ex;
    carry += tot;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

// SUMMED: sums holds the exclusive prefix of the tile sums, else the sums.
// (in and out may be one array: a thread reads its elements before it writes.)
template <bool SUMMED>
__global__ void __launch_bounds__(SCAN_THREADS) k_scan_apply(const uint32_t* in, uint64_t n, const uint32_t* limit,
                                                             bool wide, const uint32_t* __restrict__ sums,
                                                             uint32_t* out) {
  __shared__ uint32_t sm[SCAN_THREADS / WAVE], sp[SCAN_THREADS / WAVE];
  n = scan_length(n, limit);
  if ((uint64_t)blockIdx.x * SCAN_TILE >= n) {
    if (n == 0 && blockIdx.x == 0 && threadIdx.x == 0) out[0] = 0u;
    return;
  }
  const uint64_t base = (uint64_t)blockIdx.x * SCAN_TILE + (uint64_t)threadIdx.x * SCAN_ITEMS;
  uint32_t v[SCAN_ITEMS], s = 0, before = 0;
  scan_load(in, base, n, wide, v);
  if (!SUMMED)
    for (uint32_t t = threadIdx.x; t < blockIdx.x; t += SCAN_THREADS) before += sums[t];
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) s += v[k];
  uint32_t tot, lead;
  uint32_t run = block_excl_scan(s, sm, &tot);
  if (SUMMED) {
    lead = sums[blockIdx.x];
  } else {
    block_excl_scan(before, sp, &lead);
    if (blockIdx.x == (n - 1) / SCAN_TILE && threadIdx.x == 0) out[n] = lead + tot;
  }
  run += lead;
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k) {
    const uint32_t x = v[k];
    v[k] = run;
    run += x;
  }
  if (wide && base + SCAN_ITEMS <= n) {
    *(uint4*)(out + base) = make_uint4(v[0], v[1], v[2], v[3]);
    *(uint4*)(out + base + 4) = make_uint4(v[4], v[5], v[6], v[7]);
    return;
  }
#pragma unroll
  for (int k = 0; k < SCAN_ITEMS; ++k)
    if (base + k < n) out[base + k] = v[k];
}

// Short arrays (the cells of a single packing): one workgroup of 1024
// threads walks the array in tiles of 4096 with a running carry, in one
// launch.
constexpr int SCAN1_THREADS = 1024;
constexpr int SCAN1_ITEMS = 4;
constexpr uint64_t SCAN1_MAX = 16384;
__global__ void __launch_bounds__(SCAN1_THREADS) k_scan_one(const uint32_t* __restrict__ in,
                                                            uint64_t n, uint32_t* __restrict__ out) {
  __shared__ uint32_t sm[SCAN1_THREADS / WAVE];
  const int lane = threadIdx.x & (WAVE - 1);
  const int wv = threadIdx.x / WAVE;
  uint32_t carry = 0;
  for (uint64_t t0 = 0; t0 < n; t0 += (uint64_t)SCAN1_THREADS * SCAN1_ITEMS) {
    const uint64_t base = t0 + (uint64_t)threadIdx.x * SCAN1_ITEMS;
    uint32_t v[SCAN1_ITEMS];
    uint32_t sum = 0;
#pragma unroll
    for (int k = 0; k < SCAN1_ITEMS; ++k) {
      const uint64_t i = base + k;
      const uint32_t x = in[i < n ? i : n - 1];  // clamped load, masked below
      v[k] = i < n ? x : 0u;
      sum += v[k];
    }
    const uint32_t inc = wave_incl_scan(sum);
    if (lane == WAVE - 1) sm[wv] = inc;
    __syncthreads();
    uint32_t off = 0, tot = 0;
#pragma unroll
    for (int w = 0; w < SCAN1_THREADS / WAVE; ++w) {
      const uint32_t x = sm[w];
      off += w < wv ? x : 0u;
      tot += x;
    }
    __syncthreads();
    uint32_t run = carry + off + inc - sum;
#pragma unroll
    for (int k = 0; k < SCAN1_ITEMS; ++k) {
      const uint64_t i = base + k;
      if (i < n) out[i] = run;
      run += v[k];
    }
    carry += tot;
  }
  if (threadIdx.x == 0) out[n] = carry;
}

size_t scan_tmp_words(uint64_t n) { return (size_t)((n + SCAN_TILE - 1) / SCAN_TILE) + 1; }

// out[0..n) = exclusive prefix of in, out[n] = total.  in and out may alias.
// limit (optional, device): a smaller n that only the device knows; what lies
// past it is neither read (but by the one workgroup of a short array) nor
// written to any purpose.
void scan_u32(const uint32_t* in, uint32_t* out, uint64_t n, uint32_t* tmp, hipStream_t s, const uint32_t* limit) {
  if (n > 0 && n <= SCAN1_MAX) {
    hipLaunchKernelGGL(k_scan_one, dim3(1), dim3(SCAN1_THREADS), 0, s, in, n, out);
    return;
  }
  const uint32_t nt = (uint32_t)((n + SCAN_TILE - 1) / SCAN_TILE);
  if (nt == 0) {
    hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_THREADS), 0, s, tmp, 0u, out, (uint64_t)0, nullptr);
    return;
  }
  const bool wide = (((uintptr_t)in | (uintptr_t)out) & 15u) == 0;
  hipLaunchKernelGGL(k_scan_tiles, dim3(nt), dim3(SCAN_THREADS), 0, s, in, n, limit, wide, tmp);
  if (nt <= SUMS_MAX) {
    hipLaunchKernelGGL(k_scan_apply<false>, dim3(nt), dim3(SCAN_THREADS), 0, s, in, n, limit, wide, tmp, out);
    return;
  }
  hipLaunchKernelGGL(k_scan_sums, dim3(1), dim3(SCAN_THREADS), 0, s, tmp, nt, out, n, limit);
  hipLaunchKernelGGL(k_scan_apply<true>, dim3(nt), dim3(SCAN_THREADS), 0, s, in, n, limit, wide, tmp, out);
}

__global__ void k_fill_u32(uint32_t* __restrict__ p, uint32_t v, uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x)
    p[i] = v;
}

void fill_u32(uint32_t* p, uint32_t v, uint64_t n, hipStream_t s) {
  if (n == 0) return;
  uint64_t blocks = (n + 255) / 256;
  if (blocks > 4096) blocks = 4096;
  hipLaunchKernelGGL(k_fill_u32, dim3((uint32_t)blocks), dim3(256), 0, s, p, v, n);
}

}  // namespace nf
