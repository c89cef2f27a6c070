// nf_post.hip - cell-list build for a given packing, canonical ordering of
// contact rows, and exact int64 histograms.
#include "nf_internal.h"

namespace nf {

static int grid_for(uint64_t n, int threads) {
  uint64_t b = (n + threads - 1) / threads;
  if (b > 8192) b = 8192;
  if (b < 1) b = 1;
  return (int)b;
}

// ---------------------------------------------------------------------------
// Cell list of a packing (the role of writeGlbMem's per-cell placement,
// inc/memoryIO.h:361-429, for an existing packing) as a two-level counting
// sort with no device-scope atomics: those resolve beyond the XCD's L2 and
// cap a one-atomic-per-rod binning at a few tens of G/s.  Buckets are runs
// of 2^shift consecutive cells in linear cell order, so a bucket's cells
// own one contiguous range of the output.
//   1. k_bin_count: each block counts its chunk of rods per bucket in LDS
//      and writes its column of the bucket-major matrix M[bucket][block];
//   2. scan_u32 of M gives each (bucket, block) its range in bucket order;
//   3. k_bin_scatter: each block places its rods there (LDS cursors);
//   4. k_bin_cells: one workgroup per bucket counts its rods per cell in
//      LDS, scans the counts, writes the cells' start, count and largest
//      half length, and places the rods in cell order.
// The order of the rods inside a cell is not fixed (LDS atomics); every
// pass reading the list is independent of it.
// ---------------------------------------------------------------------------
constexpr int BIN_THREADS = 1024;

struct BinArg {
  int32_t nc[3];
  double sc[3];
  uint32_t shift;  // log2 of the cells per bucket
  uint32_t nb;     // buckets
  uint32_t nblk;   // blocks of passes 1 and 3
  uint32_t chunk;  // rods per block of passes 1 and 3
  uint32_t ncells;
};

__global__ void __launch_bounds__(BIN_THREADS) k_bin_count(const float4* __restrict__ P, uint32_t n, BinArg g,
                                                           uint32_t* __restrict__ M) {
  extern __shared__ uint32_t hist[];
  for (uint32_t b = threadIdx.x; b < g.nb; b += BIN_THREADS) hist[b] = 0u;
  __syncthreads();
  const uint64_t lo = (uint64_t)blockIdx.x * g.chunk;
  const uint64_t hi = lo + g.chunk < (uint64_t)n ? lo + g.chunk : (uint64_t)n;
  for (uint64_t i = lo + threadIdx.x; i < hi; i += BIN_THREADS)
    atomicAdd(&hist[cell_index(P[i], g.nc, g.sc) >> g.shift], 1u);
  __syncthreads();
  for (uint32_t b = threadIdx.x; b < g.nb; b += BIN_THREADS)
    M[(uint64_t)b * g.nblk + blockIdx.x] = hist[b];
}

__global__ void __launch_bounds__(BIN_THREADS) k_bin_scatter(const float4* __restrict__ P,
                                                             const float4* __restrict__ D, uint32_t n,
                                                             BinArg g, const uint32_t* __restrict__ M,
                                                             float4* __restrict__ tP, float4* __restrict__ tD,
                                                             uint32_t* __restrict__ tid) {
  extern __shared__ uint32_t cur[];
  for (uint32_t b = threadIdx.x; b < g.nb; b += BIN_THREADS) cur[b] = M[(uint64_t)b * g.nblk + blockIdx.x];
  __syncthreads();
  const uint64_t lo = (uint64_t)blockIdx.x * g.chunk;
  const uint64_t hi = lo + g.chunk < (uint64_t)n ? lo + g.chunk : (uint64_t)n;
  for (uint64_t i = lo + threadIdx.x; i < hi; i += BIN_THREADS) {
    const float4 p = P[i];
    const uint32_t dst = atomicAdd(&cur[cell_index(p, g.nc, g.sc) >> g.shift], 1u);
    tP[dst] = p;
    tD[dst] = D[i];
    tid[dst] = (uint32_t)i;
  }
}

__global__ void __launch_bounds__(BIN_THREADS) k_bin_cells(const float4* __restrict__ tP,
                                                           const float4* __restrict__ tD,
                                                           const uint32_t* __restrict__ tid, BinArg g,
                                                           const uint32_t* __restrict__ M,
                                                           float4* __restrict__ oP, float4* __restrict__ oD,
                                                           uint32_t* __restrict__ oid,
                                                           uint32_t* __restrict__ start,
                                                           uint32_t* __restrict__ count,
                                                           float* __restrict__ hl) {
  extern __shared__ uint32_t lds[];
  const uint32_t K = 1u << g.shift;
  uint32_t* cnt = lds;      // rods per cell
  uint32_t* mx = lds + K;   // largest half length per cell (float bits, >= 0)
  uint32_t* off = mx + K;   // exclusive prefix, then the placement cursor
  __shared__ uint32_t wsum[BIN_THREADS / WAVE];
  const uint32_t b = blockIdx.x;
  const uint32_t base = M[(uint64_t)b * g.nblk];
  const uint32_t end = M[(uint64_t)(b + 1) * g.nblk];
  const uint32_t c0 = b << g.shift;
  for (uint32_t k = threadIdx.x; k < K; k += BIN_THREADS) {
    cnt[k] = 0u;
    mx[k] = 0u;
  }
  __syncthreads();
  for (uint32_t i = base + threadIdx.x; i < end; i += BIN_THREADS) {
    const float4 p = tP[i];
    const uint32_t k = cell_index(p, g.nc, g.sc) - c0;
    atomicAdd(&cnt[k], 1u);
    atomicMax(&mx[k], __float_as_uint(p.w));
  }
  __syncthreads();
  // exclusive scan of cnt: each thread sums a run of K / BIN_THREADS cells
  // (at least one), then a wave scan and the wave totals
  const uint32_t per = (K + BIN_THREADS - 1) / BIN_THREADS;
  const uint32_t k0 = threadIdx.x * per;
  uint32_t sum = 0;
  for (uint32_t k = k0; k < k0 + per && k < K; ++k) sum += cnt[k];
  const int lane = threadIdx.x & (WAVE - 1);
  uint32_t inc = sum;
#pragma unroll
  for (int o = 1; o < WAVE; o <<= 1) {
    const uint32_t t = __shfl_up(inc, o, WAVE);
    inc += lane >= o ? t : 0u;
  }
  if (lane == WAVE - 1) wsum[threadIdx.x / WAVE] = inc;
  __syncthreads();
  uint32_t run = inc - sum;
  for (int w = 0; w < (int)(threadIdx.x / WAVE); ++w) run += wsum[w];
  for (uint32_t k = k0; k < k0 + per && k < K; ++k) {
    off[k] = run;
    run += cnt[k];
  }
  __syncthreads();
  for (uint32_t k = threadIdx.x; k < K; k += BIN_THREADS) {
    const uint32_t c = c0 + k;
    if (c < g.ncells) {
      start[c] = base + off[k];
      count[c] = cnt[k];
      hl[c] = __uint_as_float(mx[k]);
    }
  }
  if (b + 1 == g.nb && threadIdx.x == 0) start[g.ncells] = end;
  __syncthreads();
  for (uint32_t i = base + threadIdx.x; i < end; i += BIN_THREADS) {
    const float4 p = tP[i];
    const uint32_t dst = base + atomicAdd(&off[cell_index(p, g.nc, g.sc) - c0], 1u);
    oP[dst] = p;
    oD[dst] = tD[i];
    oid[dst] = tid[i];
  }
}

// Buckets of 2^shift cells, shift the smallest with at most BIN_BUCKETS
// buckets (at least 32 cells, at most 4096: 48 KB of LDS per bucket
// workgroup), and about BIN_BLOCKS blocks of at least 2048 rods for the
// histogram and scatter passes, so that each (bucket, block) range written
// by the scatter holds a few tens of rods.
constexpr uint32_t BIN_BUCKETS = 1024;
constexpr uint32_t BIN_BLOCKS = 256;

BinPlan bin_plan(uint32_t n, uint64_t ncells) {
  BinPlan bp{};
  uint32_t shift = 5;
  while (shift < 12 && ((ncells + (1ull << shift) - 1) >> shift) > BIN_BUCKETS) ++shift;
  bp.shift = shift;
  bp.nb = (uint32_t)((ncells + (1ull << shift) - 1) >> shift);
  uint64_t chunk = ((uint64_t)n + BIN_BLOCKS - 1) / BIN_BLOCKS;
  if (chunk < 2048) chunk = 2048;
  chunk = (chunk + BIN_THREADS - 1) / BIN_THREADS * BIN_THREADS;
  bp.chunk = (uint32_t)chunk;
  bp.nblk = n == 0 ? 0u : (uint32_t)(((uint64_t)n + chunk - 1) / chunk);
  bp.m_words = (uint64_t)bp.nb * bp.nblk;
  return bp;
}

void launch_bin_rods(const BinPlan& bp, const float4* P, const float4* D, uint32_t n, const int32_t ncell[3],
                     const double scale[3], uint32_t* M, uint32_t* scan_tmp, float4* tP, float4* tD,
                     uint32_t* tid, float4* oP, float4* oD, uint32_t* oid, uint32_t* start, uint32_t* count,
                     float* hl, hipStream_t s) {
  BinArg g;
  for (int a = 0; a < 3; ++a) {
    g.nc[a] = ncell[a];
    g.sc[a] = scale[a];
  }
  g.shift = bp.shift;
  g.nb = bp.nb;
  g.nblk = bp.nblk;
  g.chunk = bp.chunk;
  g.ncells = (uint32_t)((uint64_t)ncell[0] * ncell[1] * ncell[2]);
  if (n == 0) {
    fill_u32(start, 0u, (uint64_t)g.ncells + 1, s);
    fill_u32(count, 0u, g.ncells, s);
    fill_u32((uint32_t*)hl, 0u, g.ncells, s);
    return;
  }
  const size_t hist_bytes = sizeof(uint32_t) * bp.nb;
  hipLaunchKernelGGL(k_bin_count, dim3(bp.nblk), dim3(BIN_THREADS), hist_bytes, s, P, n, g, M);
  scan_u32(M, M, bp.m_words, scan_tmp, s);
  hipLaunchKernelGGL(k_bin_scatter, dim3(bp.nblk), dim3(BIN_THREADS), hist_bytes, s, P, D, n, g, M, tP, tD,
                     tid);
  hipLaunchKernelGGL(k_bin_cells, dim3(bp.nb), dim3(BIN_THREADS), sizeof(uint32_t) * 3u * (1u << bp.shift), s,
                     tP, tD, tid, g, M, oP, oD, oid, start, count, hl);
}

// ---------------------------------------------------------------------------
// Contact rows: sort each row by (J, image) so the list is canonical whatever
// order the record pass found the pairs in.  Rows are short (a few entries),
// so one thread per row with an insertion sort in global memory.
// ---------------------------------------------------------------------------
__device__ __forceinline__ bool img_less(int32_t a, int32_t b) {
#pragma unroll
  for (int d = 0; d < 3; ++d) {
    const int x = (int)(int8_t)((a >> (8 * d)) & 0xFF);
    const int y = (int)(int8_t)((b >> (8 * d)) & 0xFF);
    if (x != y) return x < y;
  }
  return false;
}

__global__ void k_row_sort(const uint32_t* __restrict__ rowptr, uint32_t n, uint32_t* __restrict__ J,
                           float* __restrict__ gap, double* __restrict__ gap64,
                           int32_t* __restrict__ img) {
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    const uint32_t b = rowptr[r], e = rowptr[r + 1];
    for (uint32_t i = b + 1; i < e; ++i) {
      const uint32_t kj = J[i];
      const int32_t ki = img[i];
      const float kg = gap[i];
      const double kd = gap64[i];
      uint32_t k = i;
      while (k > b && (J[k - 1] > kj || (J[k - 1] == kj && img_less(ki, img[k - 1])))) {
        J[k] = J[k - 1];
        img[k] = img[k - 1];
        gap[k] = gap[k - 1];
        gap64[k] = gap64[k - 1];
        --k;
      }
      J[k] = kj;
      img[k] = ki;
      gap[k] = kg;
      gap64[k] = kd;
    }
  }
}

void launch_row_sort(const uint32_t* rowptr, uint32_t n, uint32_t* J, float* gap, double* gap64,
                     int32_t* img, hipStream_t s) {
  hipLaunchKernelGGL(k_row_sort, dim3(grid_for(n, 256)), dim3(256), 0, s, rowptr, n, J, gap,
                     gap64, img);
}

// Contact area of every contact, one thread per contact: a thread per row had
// most lanes of a wave wait for the few rows that hold any (215,000 contacts of
// 4M rods 104 us, now 24; 46,000 of 500,000 rods 23 and 7, 2,000 rods 11 and 4).
__global__ void k_contact_area(const float4* __restrict__ P, const float4* __restrict__ D, uint64_t c,
                               const uint32_t* __restrict__ I, const uint32_t* __restrict__ J,
                               const int32_t* __restrict__ img, double bx, double by, double bz,
                               double rlim, double* __restrict__ area) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < c; k += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t i = I[k], j = J[k];
    const int32_t m = img[k];
    const double sx = (double)(int)(int8_t)(m & 0xFF) * bx;
    const double sy = (double)(int)(int8_t)((m >> 8) & 0xFF) * by;
    const double sz = (double)(int)(int8_t)((m >> 16) & 0xFF) * bz;
    area[k] = contact_area_f64(P[i], D[i], P[j], D[j], sx, sy, sz, rlim);
  }
}

void launch_contact_area(const float4* P, const float4* D, uint64_t c, const uint32_t* I, const uint32_t* J,
                         const int32_t* img, const double box[3], double rlim, double* area, hipStream_t s) {
  if (c == 0) return;
  hipLaunchKernelGGL(k_contact_area, dim3(grid_for(c, 256)), dim3(256), 0, s, P, D, c, I, J, img, box[0], box[1],
                     box[2], rlim, area);
}

// CSR over I from the unsorted contact list (the pair pass appends in any
// order, the row sort makes every row canonical afterwards; a row's places are
// taken from its count downwards).
__global__ void k_csr_count(const uint32_t* __restrict__ I, uint64_t c, uint32_t* __restrict__ cnt) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < c;
       k += (uint64_t)gridDim.x * blockDim.x)
    atomicAdd(&cnt[I[k]], 1u);
}

__global__ void k_csr_scatter(const uint32_t* __restrict__ I, const uint32_t* __restrict__ J,
                              const float* __restrict__ gap, const double* __restrict__ gap64,
                              const int32_t* __restrict__ img, uint64_t c,
                              const uint32_t* __restrict__ rowptr, uint32_t* __restrict__ cnt,
                              uint32_t* __restrict__ oI, uint32_t* __restrict__ oJ, float* __restrict__ ogap,
                              double* __restrict__ ogap64, int32_t* __restrict__ oimg) {
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < c;
       k += (uint64_t)gridDim.x * blockDim.x) {
    const uint32_t i = I[k];
    const uint32_t pos = rowptr[i] + atomicSub(&cnt[i], 1u) - 1u;
    oI[pos] = i;
    oJ[pos] = J[k];
    ogap[pos] = gap[k];
    ogap64[pos] = gap64[k];
    oimg[pos] = img[k];
  }
}

void launch_csr_count(const uint32_t* I, uint64_t c, uint32_t* cnt, hipStream_t s) {
  if (c == 0) return;
  hipLaunchKernelGGL(k_csr_count, dim3(grid_for(c, 256)), dim3(256), 0, s, I, c, cnt);
}

void launch_csr_scatter(const uint32_t* I, const uint32_t* J, const float* gap, const double* gap64,
                        const int32_t* img, uint64_t c, const uint32_t* rowptr, uint32_t* cnt,
                        uint32_t* oI, uint32_t* oJ, float* ogap, double* ogap64, int32_t* oimg, hipStream_t s) {
  if (c == 0) return;
  hipLaunchKernelGGL(k_csr_scatter, dim3(grid_for(c, 256)), dim3(256), 0, s, I, J, gap, gap64, img, c,
                     rowptr, cnt, oI, oJ, ogap, ogap64, oimg);
}

// ---------------------------------------------------------------------------
// Centre-centre distance statistics (statKernel_CENT, inc/statKernel_CENT.h:
// 8-122, driven by collectStats, src/statistics_collection.cu:866-1033):
// every unordered pair of distinct rods over all periodic images with centre
// distance below bins * width, binned by comparing d^2 with the squared bin
// edges, plus exact fixed-point sums of round(d 2^24) and round(d^2 2^16).
// The FP64 distance is evaluated with the lower id first and the image applied
// to the higher id, so every bin decision matches a sequential evaluation.
//
// A wave takes an item: some rods of one cell against one run of neighbour
// cells.  Cells along x follow each other in the cell list, so the half stencil
// is a few runs (five at an edge of rmax) and a run's rods are loaded 64 at a
// time, one per lane, whatever the single cells hold; the probes are uniform
// and come through scalar loads.  Of the candidates 15 % are pairs: an FP32
// test with a safe margin picks them, a queue in LDS collects 64 before the
// FP64 distance, bin and sums are evaluated, so those run with every lane.  A
// block keeps its counts and sums and writes them once; a second kernel adds
// the blocks' (atomics on the few lines of the result had cost as much as the
// pairs: 12 ns each on one line).  300,000 rods, 20 M pairs in 64 bins:
// 1313 -> 213 + 9 us, bound by FP32 and FP64 instruction issue; two or four
// probes to a look at the queue took 227 and 242 (its room costs occupancy).
// ---------------------------------------------------------------------------
constexpr int CENT_MAX_BINS = 1024;
constexpr int CENT_THREADS = 256;
constexpr int CENT_QUEUE = 2 * WAVE;

// wave-uniform copies (SGPR) of values every lane already agrees on, so the
// loops that hold barriers have scalar trip counts
__device__ __forceinline__ uint32_t uni_u32(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}

struct CentArg {
  const uint32_t* X;  // rod ids
  const uint32_t* start;
  const uint32_t* count;
  const uint32_t* cells;  // their number, then the cells that hold rods; null: every cell
  const int4* runs;  // first and last x offset, y and z offset
  uint32_t n_runs, chunks, chunk;  // a cell's rods in `chunks` shares of `chunk` at a time
  int32_t nc[3];
  double box[3];
  const double* e2;      // bins + 1 squared edges
  int bins;
  float r2f;             // FP32 prefilter bound
  float inv_width;
};

struct CentQueue {
  uint32_t p[CENT_QUEUE], q[CENT_QUEUE], img[CENT_QUEUE];
};

struct CentAcc {
  unsigned long long cnt, sq, s2q;
};

// The pair of queue entry k: its bin and its fixed-point sums.
__device__ void cent_pair(const float4* __restrict__ P, const CentArg& a, const CentQueue& L, uint32_t k,
                          const double* e2, uint32_t* hist, CentAcc& acc) {
  const uint32_t p = L.p[k], q = L.q[k], code = L.img[k];
  if (p == q) return;  // a rod and its own image
  const bool swap = a.X[p] > a.X[q];
  const float4 Pa = swap ? P[q] : P[p], Pb = swap ? P[p] : P[q];
  const int s = swap ? -1 : 1;
  const double ux = (double)(s * ((int)(code & 1023u) - 512)) * a.box[0];
  const double uy = (double)(s * ((int)((code >> 10) & 1023u) - 512)) * a.box[1];
  const double uz = (double)(s * ((int)(code >> 20) - 512)) * a.box[2];
  const double dx = ((double)Pa.x - (double)Pb.x) - ux;
  const double dy = ((double)Pa.y - (double)Pb.y) - uy;
  const double dz = ((double)Pa.z - (double)Pb.z) - uz;
  const double d2 = dx * dx + dy * dy + dz * dz;
  if (!(d2 < e2[a.bins])) return;
  // a first guess in FP32, then the edges themselves decide
  const float df = (float)d2, rf = __builtin_amdgcn_rsqf(df);
  int b = (int)fminf(df * rf * a.inv_width, (float)(a.bins - 1));
  while (b > 0 && e2[b] > d2) --b;
  while (e2[b + 1] <= d2) ++b;
  atomicAdd(&hist[b], 1u);
  ++acc.cnt;
  // round(d 2^24): one Newton step on the FP32 root is good to 2^-44 of d,
  // which settles the rounding unless the value lies within 2^-42 of a half
  const double y0 = d2 * (double)rf;
  const double y = fma(fma(-y0, y0, d2), 0.5 * (double)rf, y0);
  const double v = y * 16777216.0 + 0.5;
  double w = floor(v);
  const double f = v - w, g = v * 2.2737367544323206e-13;
  if (!(f > g && f < 1.0 - g)) w = floor(sqrt_cr(d2) * 16777216.0 + 0.5);
  acc.sq += (unsigned long long)w;
  acc.s2q += (unsigned long long)floor(d2 * 65536.0 + 0.5);
}

__global__ void __launch_bounds__(CENT_THREADS) k_cent(const float4* __restrict__ P, CentArg a,
                                                       unsigned long long* __restrict__ part) {
  __shared__ double e2[CENT_MAX_BINS + 1];
  __shared__ uint32_t hist[CENT_MAX_BINS];
  __shared__ CentQueue queue[CENT_THREADS / WAVE];
  __shared__ unsigned long long tot[3];
  for (int k = threadIdx.x; k <= a.bins; k += CENT_THREADS) {
    e2[k] = a.e2[k];
    if (k < a.bins) hist[k] = 0u;
  }
  if (threadIdx.x < 3) tot[threadIdx.x] = 0ull;
  __syncthreads();
  const uint32_t lane = threadIdx.x % WAVE, wave = uni_u32(threadIdx.x / WAVE);
  CentQueue& L = queue[wave];
  CentAcc acc = {0ull, 0ull, 0ull};
  uint32_t qn = 0u;
  const uint32_t per_cell = a.n_runs * a.chunks;
  const uint64_t items =
      (a.cells ? (uint64_t)uni_u32(a.cells[0]) : (uint64_t)a.nc[0] * (uint64_t)a.nc[1] * (uint64_t)a.nc[2]) * per_cell;
  for (uint64_t t = blockIdx.x * (CENT_THREADS / WAVE) + wave; t < items; t += gridDim.x * (CENT_THREADS / WAVE)) {
    const uint32_t at = uni_u32((uint32_t)(t / per_cell)), part_of = uni_u32((uint32_t)(t % per_cell));
    const uint32_t cell = a.cells ? uni_u32(a.cells[at + 1u]) : at;
    const uint32_t c = part_of % a.chunks;
    const int4 run = a.runs[part_of / a.chunks];
    const uint32_t pc = uni_u32(a.count[cell]), ps = uni_u32(a.start[cell]);
    if (c * a.chunk >= pc) continue;
    const int c0 = (int)(cell % (uint32_t)a.nc[0]);
    const int c1 = (int)((cell / (uint32_t)a.nc[0]) % (uint32_t)a.nc[1]) + run.z;
    const int c2 = (int)(cell / ((uint32_t)a.nc[0] * (uint32_t)a.nc[1])) + run.w;
    const int i1 = floor_div(c1, a.nc[1]), i2 = floor_div(c2, a.nc[2]);
    const uint32_t row = (uint32_t)a.nc[0] * (uint32_t)((c1 - i1 * a.nc[1]) + a.nc[1] * (c2 - i2 * a.nc[2]));
    const float fy = (float)((double)i1 * a.box[1]), fz = (float)((double)i2 * a.box[2]);
    for (int x = c0 + run.x; x <= c0 + run.y;) {
      // the part of the run in one image of the box
      const int i0 = floor_div(x, a.nc[0]), m0 = x - i0 * a.nc[0];
      const int len = min(c0 + run.y - x + 1, a.nc[0] - m0);
      const uint32_t last = row + (uint32_t)(m0 + len - 1);
      const uint32_t q0 = uni_u32(a.start[row + (uint32_t)m0]);
      const uint32_t q1 = uni_u32(a.start[last]) + uni_u32(a.count[last]);
      const bool own = run.z == 0 && run.w == 0 && x == c0;  // each pair of the cell's own rods once
      const float fx = (float)((double)i0 * a.box[0]);
      const uint32_t code = (uint32_t)(i0 + 512) | ((uint32_t)(i1 + 512) << 10) | ((uint32_t)(i2 + 512) << 20);
      for (uint32_t tb = q0; tb < q1; tb += WAVE) {
        const uint32_t q = tb + lane;
        const float4 P2 = P[min(q, q1 - 1u)];
        const float tx = q < q1 ? P2.x + fx : 3e38f, ty = P2.y + fy, tz = P2.z + fz;
        for (uint32_t pb = c * a.chunk; pb < pc; pb += a.chunks * a.chunk) {
          const uint32_t pe = min(pb + a.chunk, pc);
          for (uint32_t j = pb; j < pe; ++j) {
            const float4 P1 = P[ps + j];
            const float wx = P1.x - tx, wy = P1.y - ty, wz = P1.z - tz;
            bool hit = fmaf(wz, wz, fmaf(wy, wy, wx * wx)) <= a.r2f;
            if (own) hit = hit && q > ps + j;
            const unsigned long long m = __ballot(hit);
            if (m == 0ull) continue;
            if (hit) {
              const uint32_t at = qn + __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32),
                                                                 __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
              L.p[at] = ps + j;
              L.q[at] = q;
              L.img[at] = code;
            }
            qn += (uint32_t)__popcll(m);
            if (qn >= (uint32_t)WAVE) {
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
              qn -= WAVE;
              cent_pair(P, a, L, qn + lane, e2, hist, acc);
              __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
            }
          }
        }
      }
      x += len;
    }
  }
  __builtin_amdgcn_fence(__ATOMIC_ACQ_REL, "wavefront");
  if (lane < qn) cent_pair(P, a, L, lane, e2, hist, acc);
  acc.cnt = wave_sum_u64(acc.cnt);
  acc.sq = wave_sum_u64(acc.sq);
  acc.s2q = wave_sum_u64(acc.s2q);
  if (lane == 0u) {
    atomicAdd(&tot[0], acc.cnt);
    atomicAdd(&tot[1], acc.sq);
    atomicAdd(&tot[2], acc.s2q);
  }
  __syncthreads();
  part += (uint64_t)blockIdx.x * (a.bins + 3);
  for (int k = threadIdx.x; k < a.bins + 3; k += CENT_THREADS) part[k] = k < a.bins ? hist[k] : tot[k - a.bins];
}

// Adds the blocks' counts and sums: a lane per word, a wave per share of the blocks.
__global__ void __launch_bounds__(CENT_THREADS) k_cent_total(const unsigned long long* __restrict__ part, uint32_t nb,
                                                             uint32_t words, unsigned long long* __restrict__ out) {
  const uint32_t k = blockIdx.x * WAVE + threadIdx.x % WAVE;
  if (k >= words) return;
  unsigned long long s = 0;
#pragma unroll 4
  for (uint32_t b = blockIdx.y * (CENT_THREADS / WAVE) + threadIdx.x / WAVE; b < nb;
       b += gridDim.y * (CENT_THREADS / WAVE))
    s += part[(uint64_t)b * words + k];
  if (s) atomicAdd(&out[k], s);
}

// Rods in their cells, summed over the rods.
__global__ void __launch_bounds__(CENT_THREADS) k_cent_crowd(const uint32_t* __restrict__ count, uint64_t ncells,
                                                             unsigned long long* __restrict__ out) {
  unsigned long long s = 0;
  for (uint64_t c = (uint64_t)blockIdx.x * CENT_THREADS + threadIdx.x; c < ncells; c += (uint64_t)gridDim.x * CENT_THREADS)
    s += (unsigned long long)count[c] * count[c];
  s = wave_sum_u64(s);
  if (threadIdx.x % WAVE == 0 && s) atomicAdd(out, s);
}

void launch_cent_crowd(const uint32_t* count, uint64_t ncells, unsigned long long* out, hipStream_t s) {
  hipLaunchKernelGGL(k_cent_crowd, dim3(std::min(grid_for(ncells, 4 * CENT_THREADS), 64)), dim3(CENT_THREADS), 0, s, count,
                     ncells, out);
}

// The cells that hold rods: a block takes the places of its own with one atomic.
__global__ void __launch_bounds__(CENT_THREADS) k_cent_cells(const uint32_t* __restrict__ count, uint64_t ncells,
                                                             uint32_t* __restrict__ cells) {
  __shared__ uint32_t sh[CENT_THREADS / WAVE], base;
  const uint32_t lane = threadIdx.x % WAVE, wave = threadIdx.x / WAVE;
  for (uint64_t c0 = (uint64_t)blockIdx.x * CENT_THREADS; c0 < ncells; c0 += (uint64_t)gridDim.x * CENT_THREADS) {
    const uint64_t c = c0 + threadIdx.x;
    const bool some = c < ncells && count[c] != 0u;
    const unsigned long long m = __ballot(some);
    if (lane == 0) sh[wave] = (uint32_t)__popcll(m);
    __syncthreads();
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < CENT_THREADS / WAVE; ++w) {
      before += w < wave ? sh[w] : 0u;
      all += sh[w];
    }
    if (threadIdx.x == 0 && all) base = atomicAdd(&cells[0], all);
    __syncthreads();
    if (some) cells[1u + base + before + (uint32_t)__popcll(m & ((1ull << lane) - 1ull))] = (uint32_t)c;
  }
}

void launch_cent_cells(const uint32_t* count, uint64_t ncells, uint32_t* cells, hipStream_t s) {
  fill_u32(cells, 0u, 1, s);
  hipLaunchKernelGGL(k_cent_cells, dim3(grid_for(ncells, CENT_THREADS)), dim3(CENT_THREADS), 0, s, count, ncells, cells);
}

void launch_cent(const float4* P, const uint32_t* X, const uint32_t* start, const uint32_t* count,
                 const uint32_t* cells, const int4* runs, uint32_t n_runs, double mean, const int32_t nc[3],
                 const double box[3], const double* e2, int bins, double width, float r2f, unsigned long long* part,
                 unsigned long long* out, hipStream_t s) {
  CentArg a;
  a.X = X;
  a.start = start;
  a.count = count;
  a.cells = cells;
  a.runs = runs;
  a.n_runs = n_runs;
  for (int d = 0; d < 3; ++d) {
    a.nc[d] = nc[d];
    a.box[d] = box[d];
  }
  a.e2 = e2;
  a.bins = bins;
  a.r2f = r2f;
  a.inv_width = (float)(1.0 / width);
  // shares of 32 probes, of fewer where cells and runs alone leave the chip idle
  const uint64_t cr = (uint64_t)nc[0] * nc[1] * nc[2] * n_runs;
  const uint64_t rods = (uint64_t)mean + 1;
  a.chunk = 32;
  while (a.chunk > 4 && cr * ((rods + a.chunk - 1) / a.chunk) < 16384) a.chunk /= 2;
  // (a list's cells are few among cr)
  const uint64_t most = cells ? 64 : 65536 / std::min<uint64_t>(cr, 65536);
  a.chunks = (uint32_t)std::max<uint64_t>(1, std::min<uint64_t>((rods + a.chunk - 1) / a.chunk, most));
  const int blocks = std::min(grid_for(cr * a.chunks, CENT_THREADS / WAVE), CENT_BLOCKS);
  hipLaunchKernelGGL(k_cent, dim3(blocks), dim3(CENT_THREADS), 0, s, P, a, part);
  const uint32_t words = (uint32_t)bins + 3;
  hipLaunchKernelGGL(k_cent_total, dim3((words + WAVE - 1) / WAVE, 64), dim3(CENT_THREADS), 0, s, part,
                     (uint32_t)blocks, words, out);
}

// ---------------------------------------------------------------------------
// Van der Waals energy over the sorted contact list (statKernel_VdW_naive,
// inc/statKernel_MUT.h:531-628, driven by collect_vdw,
// src/statistics_collection.cu:53-154): one thread per row sums its
// contributing pairs in row order; rows are summed in blocks of 1024 in
// order, block sums in order (deterministic).
// ---------------------------------------------------------------------------
__global__ void k_vdw_rows(const float4* __restrict__ P, const float4* __restrict__ D, uint32_t n,
                           const uint32_t* __restrict__ rowptr, const uint32_t* __restrict__ J,
                           const int32_t* __restrict__ img, double bx, double by, double bz,
                           double dlim, double A, double B, double* __restrict__ rowsum,
                           unsigned long long* __restrict__ pairs) {
  unsigned long long local = 0;
  for (uint32_t r = blockIdx.x * blockDim.x + threadIdx.x; r < n; r += gridDim.x * blockDim.x) {
    double s = 0.0;
    const float4 P1 = P[r], D1 = D[r];
    for (uint32_t k = rowptr[r]; k < rowptr[r + 1]; ++k) {
      const int32_t c = img[k];
      const double sx = (double)(int)(int8_t)(c & 0xFF) * bx;
      const double sy = (double)(int)(int8_t)((c >> 8) & 0xFF) * by;
      const double sz = (double)(int)(int8_t)((c >> 16) & 0xFF) * bz;
      double e;
      if (vdw_pair(P1, D1, P[J[k]], D[J[k]], sx, sy, sz, dlim, A, B, &e)) {
        s = s + e;
        ++local;
      }
    }
    rowsum[r] = s;
  }
  local = wave_sum_u64(local);
  if ((threadIdx.x & (WAVE - 1)) == 0 && local) atomicAdd(pairs, local);
}

__global__ void k_block_sums(const double* __restrict__ v, uint64_t n, double* __restrict__ bsum) {
  const uint64_t nb = (n + 1023) / 1024;
  for (uint64_t b = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; b < nb;
       b += (uint64_t)gridDim.x * blockDim.x) {
    const uint64_t e = (b + 1) * 1024 < n ? (b + 1) * 1024 : n;
    double s = 0.0;
    for (uint64_t k = b * 1024; k < e; ++k) s = s + v[k];
    bsum[b] = s;
  }
}

__global__ void k_block_total(const double* __restrict__ bsum, uint64_t nb, double* __restrict__ out) {
  if (blockIdx.x != 0 || threadIdx.x != 0) return;
  double t = 0.0;
  for (uint64_t b = 0; b < nb; ++b) t = t + bsum[b];
  *out = t;
}

void launch_vdw(const float4* P, const float4* D, uint32_t n, const uint32_t* rowptr,
                const uint32_t* J, const int32_t* img, const double box[3], double dlim, double A,
                double B, double* rowsum, double* bsum, double* out, unsigned long long* pairs,
                hipStream_t s) {
  if (n > 0)
    hipLaunchKernelGGL(k_vdw_rows, dim3(grid_for(n, 256)), dim3(256), 0, s, P, D, n, rowptr, J, img,
                       box[0], box[1], box[2], dlim, A, B, rowsum, pairs);
  const uint64_t nb = ((uint64_t)n + 1023) / 1024;
  if (nb > 0)
    hipLaunchKernelGGL(k_block_sums, dim3(grid_for(nb, 256)), dim3(256), 0, s, rowsum, (uint64_t)n,
                       bsum);
  hipLaunchKernelGGL(k_block_total, dim3(1), dim3(64), 0, s, bsum, nb, out);
}

// ---------------------------------------------------------------------------
// Histograms.  Angle bins by comparison with cos(bin edge): bin = number of
// edges k in 1..nb-1 with cos(angle) <= cos(edge_k), found by binary search
// on the decreasing edge table; the counts are exact (LDS u32 per block,
// then int64 atomics).  Replaces statKernel_ANGL (inc/statKernel_ANGL.h:
// 13-76) and statKernel_MUT_ANGLE_weightedFloat (inc/statKernel_MUT.h:
// 26-131) with their uint32/float accumulators.  What a block adds to the
// result bounds small packings, so there are few blocks: 300,000 rods in 1024
// of 256 threads 29 + 25 us, in 256 of 1024 15 + 12 (4M: 69 + 73, 58 + 66); the
// mutual angles by contact instead of by row 6 (13).
// ---------------------------------------------------------------------------
constexpr int HIST_THREADS = 1024;
constexpr int HIST_BLOCKS = 256;
constexpr int HIST_MAX_BINS = 256;
constexpr int HIST_MAX_2D = 4096;

__device__ __forceinline__ int edge_bin(double v, const double* __restrict__ e, int nb) {
  // largest k in [1, nb-1] with e[k] >= v, 0 if none (e decreasing)
  int lo = 0, hi = nb;  // answer in [lo, hi)
  while (hi - lo > 1) {
    const int mid = (lo + hi) >> 1;
    if (e[mid] >= v)
      lo = mid;
    else
      hi = mid;
  }
  return lo;
}

struct HistArg {
  const double* ep;
  const double* em;
  const double* et;
  const double* ephi;
  int nb, npb, ntb, axis;
  double L;
  double mu[3];
};

__global__ void __launch_bounds__(HIST_THREADS) k_hist_rods(const float4* __restrict__ P,
                                                            const float4* __restrict__ D,
                                                            uint32_t n, HistArg h,
                                                            unsigned long long* __restrict__ out) {
  __shared__ uint32_t hc[HIST_MAX_BINS], hp[HIST_MAX_BINS];
  __shared__ uint32_t h2[HIST_MAX_2D];
  const int n2 = h.npb * h.ntb;
  for (int k = threadIdx.x; k < HIST_MAX_BINS; k += blockDim.x) hc[k] = hp[k] = 0;
  for (int k = threadIdx.x; k < n2; k += blockDim.x) h2[k] = 0;
  __syncthreads();
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float4 p = P[i], d = D[i];
    const float pa = h.axis == 0 ? p.x : (h.axis == 1 ? p.y : p.z);
    const double t = (double)pa / h.L;
    int b = (int)(t * (double)h.nb);
    b = b < 0 ? 0 : (b >= h.nb ? h.nb - 1 : b);
    atomicAdd(&hc[b], 1u);
    const double cx = d.x, cy = d.y, cz = d.z;
    const double cn = sqrt_cr((cx * cx + cy * cy) + cz * cz);
    const double cosv = ((cx * h.mu[0] + cy * h.mu[1]) + cz * h.mu[2]) / cn;
    atomicAdd(&hp[edge_bin(cosv, h.ep, h.nb)], 1u);
    if (n2 > 0) {
      const double ct = cz / cn;
      const int tb = edge_bin(ct, h.et, h.ntb);
      const double rxy = sqrt_cr(cx * cx + cy * cy);
      int pb = 0;
      if (rxy > 0.0) {
        const double cp = cx / rxy;
        const int bb = edge_bin(cp, h.ephi, h.npb / 2);
        pb = cy >= 0.0 ? bb : (h.npb - 1 - bb);
      }
      atomicAdd(&h2[tb * h.npb + pb], 1u);
    }
  }
  __syncthreads();
  for (int k = threadIdx.x; k < h.nb; k += blockDim.x) {
    if (hc[k]) atomicAdd(&out[k], (unsigned long long)hc[k]);
    if (hp[k]) atomicAdd(&out[h.nb + k], (unsigned long long)hp[k]);
  }
  for (int k = threadIdx.x; k < n2; k += blockDim.x)
    if (h2[k]) atomicAdd(&out[3 * h.nb + k], (unsigned long long)h2[k]);
}

// Mutual angle of contact pairs, one thread per contact.
__global__ void __launch_bounds__(HIST_THREADS) k_hist_mut(const float4* __restrict__ D, uint64_t c,
                                                           const uint32_t* __restrict__ I,
                                                           const uint32_t* __restrict__ J,
                                                           HistArg h,
                                                           unsigned long long* __restrict__ out) {
  __shared__ uint32_t hm[HIST_MAX_BINS];
  for (int k = threadIdx.x; k < HIST_MAX_BINS; k += blockDim.x) hm[k] = 0;
  __syncthreads();
  for (uint64_t k = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; k < c; k += (uint64_t)gridDim.x * blockDim.x) {
    const float4 a = D[I[k]], b = D[J[k]];
    const double ax = a.x, ay = a.y, az = a.z, bx = b.x, by = b.y, bz = b.z;
    const double na = sqrt_cr((ax * ax + ay * ay) + az * az);
    const double nbv = sqrt_cr((bx * bx + by * by) + bz * bz);
    const double dv = fabs((ax * bx + ay * by) + az * bz) / (na * nbv);
    atomicAdd(&hm[edge_bin(dv, h.em, h.nb)], 1u);
  }
  __syncthreads();
  for (int k = threadIdx.x; k < h.nb; k += blockDim.x)
    if (hm[k]) atomicAdd(&out[2 * h.nb + k], (unsigned long long)hm[k]);
}

// out layout: [centre nb][polar nb][mutual nb][phitheta npb*ntb]
void launch_hist(const float4* P, const float4* D, uint32_t n, uint64_t n_contacts, const uint32_t* I,
                 const uint32_t* J, const double* edges_p, const double* edges_m,
                 const double* edges_t, int nb, int npb, int ntb, int axis, double L,
                 const double* mu, unsigned long long* out, hipStream_t s) {
  HistArg h;
  h.ep = edges_p;
  h.em = edges_m;
  h.et = edges_t;
  h.ephi = edges_t ? edges_t + (ntb + 1) : nullptr;
  h.nb = nb;
  h.npb = npb;
  h.ntb = ntb;
  h.axis = axis;
  h.L = L;
  for (int a = 0; a < 3; ++a) h.mu[a] = mu[a];
  const int blocks = std::min(grid_for(n, HIST_THREADS), HIST_BLOCKS);
  hipLaunchKernelGGL(k_hist_rods, dim3(blocks), dim3(HIST_THREADS), 0, s, P, D, n, h, out);
  if (I && n_contacts)
    hipLaunchKernelGGL(k_hist_mut, dim3(std::min(grid_for(n_contacts, HIST_THREADS), HIST_BLOCKS)), dim3(HIST_THREADS), 0,
                       s, D, n_contacts, I, J, h, out);
}

// ---------------------------------------------------------------------------
// Device arithmetic self-test: the FP64 building blocks whose results must be
// bit-identical to the CPU (correctly rounded sqrt, IEEE division, the
// library's exp/log, uniform conversion).
// ---------------------------------------------------------------------------
__global__ void k_selftest(int which, const double* __restrict__ in, double* __restrict__ out,
                           uint64_t n) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n;
       i += (uint64_t)gridDim.x * blockDim.x) {
    double r = 0.0;
    switch (which) {
      case 0: r = sqrt_cr(in[i]); break;
      case 1: r = dexp(in[i]); break;
      case 2: r = dlog(in[i]); break;
      case 3: r = in[2 * i] / in[2 * i + 1]; break;
      case 4: {
        const uint64_t b = __builtin_bit_cast(uint64_t, in[i]);
        r = u01((uint32_t)(b >> 32), (uint32_t)b);
        break;
      }
      case 6: r = in[i]; break;
      default: r = sqrt(in[i]); break;
    }
    out[i] = r;
  }
}

// The FP32 screen and band of one pair per thread, as the pair passes run
// them on the device: rods as 8 floats (centre, direction, length,
// radius), the FP64 image shift of rod b, the cut distance as the passes
// form it (contact: a_1 + a_2 + gap; generation: soft (a_1 + a_2) + sep).
__global__ void k_selftest_pairs(const float* __restrict__ ra, const float* __restrict__ rb,
                                 const double* __restrict__ sh, uint64_t n, int contact, double sep_or_gap,
                                 double soft_frac, float ew, int32_t* __restrict__ out_screen,
                                 int32_t* __restrict__ out_dec, int32_t* __restrict__ out_within) {
  for (uint64_t i = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (uint64_t)gridDim.x * blockDim.x) {
    const float* a = ra + 8 * i;
    const float* b = rb + 8 * i;
    const float4 P1 = make_float4(a[0], a[1], a[2], 0.5f * a[6]);
    const float4 D1 = make_float4(a[3], a[4], a[5], a[7]);
    const float4 P2 = make_float4(b[0], b[1], b[2], 0.5f * b[6]);
    const float4 D2 = make_float4(b[3], b[4], b[5], b[7]);
    const float R32 = contact ? ((D1.w + D2.w) + (float)sep_or_gap)
                              : ((float)soft_frac * (D1.w + D2.w) + (float)sep_or_gap);
    const float sx = (float)sh[3 * i], sy = (float)sh[3 * i + 1], sz = (float)sh[3 * i + 2];
    out_screen[i] = pair_f32_screen(P1, D1, P2, D2, sx, sy, sz, R32, ew);
    const F32Pair r = pair_f32(P1, D1, P2, D2, sx, sy, sz, R32, ew, !contact);
    out_dec[i] = r.decided;
    out_within[i] = r.within;
  }
}

void launch_selftest_pairs(const float* ra, const float* rb, const double* sh, uint64_t n, int contact,
                           double sep_or_gap, double soft_frac, float ew, int32_t* out_screen, int32_t* out_dec,
                           int32_t* out_within, hipStream_t s) {
  hipLaunchKernelGGL(k_selftest_pairs, dim3(grid_for(n, 256)), dim3(256), 0, s, ra, rb, sh, n, contact, sep_or_gap,
                     soft_frac, ew, out_screen, out_dec, out_within);
}

void launch_selftest(int which, const double* in, double* out, uint64_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_selftest, dim3(grid_for(n, 256)), dim3(256), 0, s, which, in, out, n);
}


// ---------------------------------------------------------------------------
// Bounds of rods given by the caller: 32 bytes read per rod (the host had read
// them back and scanned them: 1.0 ms for 200,000 rods; here 7.7 us).  One look
// at each bound per block, and an atomic only where it grows: atomics on one
// address retire at 12 ns apiece, 110 us with three per wave.
// ---------------------------------------------------------------------------
__global__ void __launch_bounds__(256) k_rod_bounds(const float4* __restrict__ P, const float4* __restrict__ D,
                                                    uint32_t n, uint32_t* __restrict__ out) {
  float hl = 0.0f, a = 0.0f, dev = 0.0f;
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float4 p = P[i], d = D[i];
    hl = fmaxf(hl, p.w);
    a = fmaxf(a, d.w);
    const float e = fabsf(fmaf(d.z, d.z, fmaf(d.y, d.y, d.x * d.x)) - 1.0f);
    dev = e <= 1e30f ? fmaxf(dev, e) : 1e30f;  // not a number, or out of range
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) {
    hl = fmaxf(hl, __shfl_xor(hl, o, WAVE));
    a = fmaxf(a, __shfl_xor(a, o, WAVE));
    dev = fmaxf(dev, __shfl_xor(dev, o, WAVE));
  }
  __shared__ float sh[3][4];
  const uint32_t w = threadIdx.x / WAVE;
  if (threadIdx.x % WAVE == 0) {
    sh[0][w] = hl;
    sh[1][w] = a;
    sh[2][w] = dev;
  }
  __syncthreads();
  if (threadIdx.x < 3) {
    const float* v = sh[threadIdx.x];
    const uint32_t m = __float_as_uint(fmaxf(fmaxf(v[0], v[1]), fmaxf(v[2], v[3])));
    if (m > __hip_atomic_load(&out[threadIdx.x], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT))
      atomicMax(&out[threadIdx.x], m);
  }
}

void launch_rod_bounds(const float4* P, const float4* D, uint32_t n, uint32_t* out, hipStream_t s) {
  if (n == 0) return;
  const int g = grid_for(n, 256);
  hipLaunchKernelGGL(k_rod_bounds, dim3(g > 1024 ? 1024 : g), dim3(256), 0, s, P, D, n, out);
}

__global__ void __launch_bounds__(256) k_to_pinned(const uint32_t* __restrict__ src, uint64_t words,
                                                   uint64_t quads, uint32_t* __restrict__ dst) {
  const uint64_t step = (uint64_t)gridDim.x * 256u;
  const uint64_t t = blockIdx.x * 256u + threadIdx.x;
  for (uint64_t k = t; k < quads; k += step) ((uint4*)dst)[k] = ((const uint4*)src)[k];
  for (uint64_t k = 4 * quads + t; k < words; k += step) dst[k] = src[k];
}

void launch_to_pinned(const void* src, size_t bytes, void* dst, hipStream_t s) {
  const uint64_t words = bytes / 4;
  if (words == 0) return;
  const uint64_t quads = ((uintptr_t)src | (uintptr_t)dst) % 16 == 0 ? words / 4 : 0;
  hipLaunchKernelGGL(k_to_pinned, dim3(grid_for(words - 3 * quads, 256)), dim3(256), 0, s, (const uint32_t*)src, words,
                     quads, (uint32_t*)dst);
}

// Rods as eight floats each, a lane per half so that a wave writes whole lines:
// `rods` is pinned host memory, and the bus bounds it.
__global__ void __launch_bounds__(256) k_pack_rods(const float4* __restrict__ P, const float4* __restrict__ D,
                                                   uint32_t n, float4* __restrict__ rods) {
  for (uint32_t t = blockIdx.x * 256u + threadIdx.x; t < 2u * n; t += gridDim.x * 256u) {
    const float4 p = P[t >> 1], d = D[t >> 1];
    rods[t] = (t & 1u) ? make_float4(d.y, d.z, 2.0f * p.w, d.w) : make_float4(p.x, p.y, p.z, d.x);
  }
}

void launch_pack_rods(const float4* P, const float4* D, uint32_t n, float4* rods, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_pack_rods, dim3(grid_for(2ull * n, 256)), dim3(256), 0, s, P, D, n, rods);
}

// ---------------------------------------------------------------------------
// expand: periodic copies of the rods near the two faces normal to axis k.
// A rod whose centre lies within B of the far face (x >= L - B) gets a copy
// below the box, one within B of the near face (x < B) a copy above it;
// every coordinate along k is then shifted by B (new box [0, L + 2B)).  The
// shifts are FP64 sums rounded once to FP32.
// ---------------------------------------------------------------------------
__global__ void k_expand_flags(const float4* __restrict__ P, uint32_t n, int k, double L, double B,
                               uint32_t* __restrict__ below, uint32_t* __restrict__ above) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float4 p = P[i];
    const double x = (double)(k == 0 ? p.x : (k == 1 ? p.y : p.z));
    below[i] = x >= L - B ? 1u : 0u;
    above[i] = x < B ? 1u : 0u;
  }
}

__device__ __forceinline__ float4 expand_shift(float4 p, int k, double s) {
  if (k == 0)
    p.x = (float)((double)p.x + s);
  else if (k == 1)
    p.y = (float)((double)p.y + s);
  else
    p.z = (float)((double)p.z + s);
  return p;
}

__global__ void k_expand_scatter(const float4* __restrict__ P, const float4* __restrict__ D, uint32_t n, int k,
                                 double L, double B, const uint32_t* __restrict__ below,
                                 const uint32_t* __restrict__ rank_below, const uint32_t* __restrict__ above,
                                 const uint32_t* __restrict__ rank_above, uint32_t n_below,
                                 float4* __restrict__ oP, float4* __restrict__ oD) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) {
    const float4 p = P[i], d = D[i];
    oP[i] = expand_shift(p, k, B);
    oD[i] = d;
    if (below[i]) {
      const uint32_t j = n + rank_below[i];
      oP[j] = expand_shift(p, k, B - L);
      oD[j] = d;
    }
    if (above[i]) {
      const uint32_t j = n + n_below + rank_above[i];
      oP[j] = expand_shift(p, k, B + L);
      oD[j] = d;
    }
  }
}

void launch_expand_flags(const float4* P, uint32_t n, int k, double L, double B, uint32_t* below, uint32_t* above,
                         hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_expand_flags, dim3(grid_for(n, 256)), dim3(256), 0, s, P, n, k, L, B, below, above);
}

void launch_expand_scatter(const float4* P, const float4* D, uint32_t n, int k, double L, double B,
                           const uint32_t* below, const uint32_t* rank_below, const uint32_t* above,
                           const uint32_t* rank_above, uint32_t n_below, float4* oP, float4* oD, hipStream_t s) {
  if (n == 0) return;
  hipLaunchKernelGGL(k_expand_scatter, dim3(grid_for(n, 256)), dim3(256), 0, s, P, D, n, k, L, B, below,
                     rank_below, above, rank_above, n_below, oP, oD);
}

}  // namespace nf
