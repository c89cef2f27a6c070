// nf_solve.hip - DC effective conductance of the Kirchhoff network between
// the two electrodes: source at potential 1, sink at 0.
//
// Replaces the solve of tools/kirchhoff/kirchhoff.py:256-272 (scipy
// spsolve or MKL DSS on diag(S) - A - A^T with the source couplings as
// right-hand side; current I = sum (1 - V_i) B_i) for the real, DC
// conductances g0 exp(-gap / lambda) of the network matrix.
//
// Only components that touch both electrodes carry current: a component
// touching one electrode sits at its potential, one touching none is
// floating.  The rods of the current-carrying components are compacted
// into a reduced system A x = b (A: the Laplacian rows restricted to those
// rods, electrode couplings kept on the diagonal; b: the source couplings),
// which is symmetric positive definite, and solved by Jacobi-preconditioned
// conjugate gradients in FP64.
//
// Every reduction is a fixed-order tree over fixed per-block ranges, so a
// solve is bit-reproducible on one device and grid.  An iteration is two
// kernels: the product (which also forms the new direction and the sum p.Ap)
// and the update (x, r, z and the sums r.z, r.r); each block of the next
// kernel adds up the block sums of the one before, so no launch serves a
// scalar alone.  On systems that stay in the caches the chain of dependent
// loads and the launches bound an iteration, on larger ones the CSR and the
// vectors that it streams.
#include <algorithm>

#include "nf_internal.h"

namespace nf {

namespace {

constexpr int NT = 256;

// x of the lane that the DPP control names, 0 where there is none.
template <int CTRL, int ROWS>
__device__ __forceinline__ double dpp_f64(double x) {
  const long long b = __double_as_longlong(x);
  const int lo = __builtin_amdgcn_update_dpp(0, (int)b, CTRL, ROWS, 0xF, false);
  const int hi = __builtin_amdgcn_update_dpp(0, (int)(b >> 32), CTRL, ROWS, 0xF, false);
  return __longlong_as_double(((long long)hi << 32) | (uint32_t)lo);
}

// Sum over a wave in a fixed order, in lane 63 (shuffles through LDS took
// three times as long, and an iteration waits for five sums in a row).
__device__ __forceinline__ double wave_sum_last(double v) {
  v += dpp_f64<0xB1, 0xF>(v);   // lane ^ 1
  v += dpp_f64<0x4E, 0xF>(v);   // lane ^ 2
  v += dpp_f64<0x141, 0xF>(v);  // the other quad of eight lanes
  v += dpp_f64<0x140, 0xF>(v);  // the other eight of a row of 16
  v += dpp_f64<0x142, 0xA>(v);  // row before, into rows 1 and 3
  v += dpp_f64<0x143, 0xC>(v);  // rows 0 and 1, into rows 2 and 3
  return v;
}

// Sums over a block of NW waves, valid in every thread: the waves' sums in
// order.  sh[NW] is written once per call.
template <int NW = NT / WAVE>
__device__ __forceinline__ double block_sum(double v, double* sh) {
  v = wave_sum_last(v);
  if (threadIdx.x % WAVE == WAVE - 1) sh[threadIdx.x / WAVE] = v;
  __syncthreads();
  double t = 0.0;
#pragma unroll
  for (int k = 0; k < NW; ++k) t += sh[k];
  return t;
}

template <int NW = NT / WAVE>
__device__ __forceinline__ double2 block_sum2(double v, double w, double2* sh) {
  v = wave_sum_last(v);
  w = wave_sum_last(w);
  if (threadIdx.x % WAVE == WAVE - 1) sh[threadIdx.x / WAVE] = make_double2(v, w);
  __syncthreads();
  double2 t = make_double2(0.0, 0.0);
#pragma unroll
  for (int k = 0; k < NW; ++k) {
    t.x += sh[k].x;
    t.y += sh[k].y;
  }
  return t;
}

// The block's place among the rows: each XCD, which takes every eighth block,
// has a stretch of its own, so that the columns of its rows (unknowns are in
// spatial order) are mostly in its stretch too and are fetched once, not by all
// eight.
__device__ __forceinline__ uint32_t row_block() {
  const uint32_t x = blockIdx.x % 8u, q = gridDim.x / 8u, r = gridDim.x % 8u;
  return x * q + min(x, r) + blockIdx.x / 8u;
}

// This thread's share of at most CG_MAX_BLOCKS block sums of an earlier
// kernel: loads without a branch, so that they go out with the caller's.
template <int NW = NT / WAVE>
__device__ __forceinline__ double part_share(const double* __restrict__ part, uint32_t nb) {
  constexpr uint32_t STEP = NW * WAVE;
  double w[CG_MAX_BLOCKS / STEP], v = 0.0;
#pragma unroll
  for (uint32_t q = 0; q < CG_MAX_BLOCKS / STEP; ++q) w[q] = part[min(threadIdx.x + q * STEP, nb - 1u)];
#pragma unroll
  for (uint32_t q = 0; q < CG_MAX_BLOCKS / STEP; ++q) v += threadIdx.x + q * STEP < nb ? w[q] : 0.0;
  return v;
}

// Marks the components coupled to the source (bit 0) and the sink (bit 1):
// the electrode rows N and N+1 list their coupled rods.
__global__ void __launch_bounds__(NT) k_cs_flag(const uint32_t* __restrict__ nrow,
                                                const uint32_t* __restrict__ ncol,
                                                const uint32_t* __restrict__ labels, uint32_t n,
                                                uint32_t* __restrict__ flag) {
  // one atomic per wave for the component of its first lane: most coupled rods
  // are of the current-carrying one, and one address takes 12 ns each time
  const uint32_t b = nrow[n], e = nrow[n + 2], mid = nrow[n + 1];
  for (uint32_t k0 = b + blockIdx.x * NT + (threadIdx.x & ~(WAVE - 1u)); k0 < e; k0 += gridDim.x * NT) {
    const uint32_t k = k0 + threadIdx.x % WAVE;
    const uint32_t j = k < e ? ncol[k] : n;
    if (j >= n) continue;
    const uint32_t l = labels[j], bit = k < mid ? 1u : 2u;
    const uint32_t first = (uint32_t)__builtin_amdgcn_readfirstlane((int)l);
    const bool src = __ballot(l == first && bit == 1u) != 0ull, snk = __ballot(l == first && bit == 2u) != 0ull;
    const unsigned long long same = __ballot(l == first);
    if (l != first)
      atomicOr(&flag[l], bit);
    else if ((threadIdx.x % WAVE) == (uint32_t)__builtin_ctzll(same))
      atomicOr(&flag[first], (src ? 1u : 0u) | (snk ? 2u : 0u));
  }
}

// act[i] = 1 for rods in components touching both electrodes; rl[i] = the
// number of rod columns in their rows (0 elsewhere).
__global__ void __launch_bounds__(NT) k_cs_active(const uint32_t* __restrict__ nrow,
                                                  const uint32_t* __restrict__ ncol,
                                                  const uint32_t* __restrict__ labels,
                                                  const uint32_t* __restrict__ flag, uint32_t n,
                                                  uint32_t* __restrict__ act,
                                                  uint32_t* __restrict__ rl) {
  for (uint32_t i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
    const bool a = flag[labels[i]] == 3u;
    uint32_t c = 0;
    if (a)
      for (uint32_t k = nrow[i]; k < nrow[i + 1]; ++k) c += ncol[k] < n ? 1u : 0u;
    act[i] = a ? 1u : 0u;
    rl[i] = c;
  }
}

// Reduced system: CSR (columns renumbered, ascending order kept), inverse
// diagonal, source and sink couplings.
__global__ void __launch_bounds__(NT) k_cs_fill(const uint32_t* __restrict__ nrow,
                                                const uint32_t* __restrict__ ncol,
                                                const double* __restrict__ nval, uint32_t n,
                                                const uint32_t* __restrict__ act,
                                                const uint32_t* __restrict__ idx,
                                                const uint32_t* __restrict__ off,
                                                uint32_t* __restrict__ crow,
                                                uint32_t* __restrict__ ccol,
                                                double* __restrict__ cval,
                                                double* __restrict__ dinv, double* __restrict__ bsrc,
                                                double* __restrict__ bsnk) {
  for (uint32_t i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
    if (!act[i]) continue;
    const uint32_t r = idx[i];
    uint32_t pos = off[i];
    crow[r] = pos;
    double gs = 0.0, gk = 0.0, dg = 1.0;
    for (uint32_t k = nrow[i]; k < nrow[i + 1]; ++k) {
      const uint32_t j = ncol[k];
      const double v = nval[k];
      if (j < n) {
        ccol[pos] = idx[j];
        cval[pos] = v;
        ++pos;
        if (j == i) dg = v;
      } else if (j == n) {
        gs = -v;
      } else {
        gk = -v;
      }
    }
    dinv[r] = 1.0 / dg;
    bsrc[r] = gs;
    bsnk[r] = gk;
  }
}

// Unknown numbering in a spatial order: ord lists the rods by cell, so
// rods that share contacts get nearby unknowns and the matrix-vector
// product's gathers stay within cached lines.  Gathers the active flags
// and row lengths into that order; the scans of them are scattered back to
// per-rod unknown indices and row offsets.
__global__ void __launch_bounds__(NT) k_cs_to_order(uint32_t n, const uint32_t* __restrict__ ord,
                                                    const uint32_t* __restrict__ act,
                                                    const uint32_t* __restrict__ rl, uint32_t* __restrict__ acto,
                                                    uint32_t* __restrict__ rlo) {
  for (uint32_t k = blockIdx.x * NT + threadIdx.x; k < n; k += gridDim.x * NT) {
    const uint32_t i = ord[k];
    acto[k] = act[i];
    rlo[k] = rl[i];
  }
}

__global__ void __launch_bounds__(NT) k_cs_from_order(uint32_t n, const uint32_t* __restrict__ ord,
                                                      const uint32_t* __restrict__ idxo,
                                                      const uint32_t* __restrict__ offo,
                                                      uint32_t* __restrict__ idx, uint32_t* __restrict__ off) {
  for (uint32_t k = blockIdx.x * NT + threadIdx.x; k <= n; k += gridDim.x * NT) {
    const uint32_t i = k < n ? ord[k] : n;  // the totals stay at n
    idx[i] = idxo[k];
    off[i] = offo[k];
  }
}

// x = 0, r = b, (z, p) = (D^-1 r, 0); partials of r.z and b.b.
__global__ void __launch_bounds__(NT) k_cg_init(CgArgs a) {
  __shared__ double2 sh[NT / WAVE];
  double rz = 0.0, bb = 0.0;
  for (uint32_t k = blockIdx.x * NT + threadIdx.x; k < a.m; k += gridDim.x * NT) {
    const double bk = a.bsrc[k], zk = a.dinv[k] * bk;
    a.x[k] = 0.0;
    a.r[k] = bk;
    a.zp[k] = make_double2(zk, 0.0);
    rz += bk * zk;
    bb += bk * bk;
  }
  const double2 t = block_sum2(rz, bb, sh);
  if (threadIdx.x == 0) {
    a.part_rz[blockIdx.x] = t.x;
    a.part_rr[blockIdx.x] = t.y;
  }
}

// p = z + beta p and q = A p; partial of p.q.  z and the last direction lie
// side by side, so a column costs one 16-byte gather and the direction needs
// no pass of its own; it is written for the update kernel, not over the last
// one, which other rows still read.
//
// Two lanes per row, lane j summing its entries j, j + 2, ...; the lane sums
// combine in a fixed order, so the result is reproducible.  A row's chain of
// dependent loads (offsets, column, gather) bounds it, not the bytes: the first
// eight entries and the block sums that beta needs are fetched side by side,
// and every row of 262,000 is in flight at once.  178,000 unknowns with 3.9
// entries a row: 6.8 us, and the update 4.5 (7.2 and 5.8 with blocks in launch
// order, see row_block), where product, direction, update
// and two scalars had been launches of 9.9, 3.5, 4.3 and 3.1 us each; 3120
// iterations 64 -> 36 ms.  One or four lanes per row: 7.2, 8.7 us (in launch order).
constexpr int SPMV_LANES = 2, SPMV_AHEAD = 8 / SPMV_LANES;  // entries of a row fetched at once: 8
constexpr int SPMV_NT = 512;
constexpr int SPMV_ROWS = SPMV_NT / SPMV_LANES;

struct SpmvRow {
  uint32_t e0, e1;
  double v[SPMV_AHEAD];
  double2 w[SPMV_AHEAD], own;
};

__device__ __forceinline__ void spmv_fetch(const CgArgs& a, uint32_t k, uint32_t sub, SpmvRow& r) {
  const uint32_t kr = min(k, a.m - 1u);
  uint32_t c[SPMV_AHEAD];
  r.e0 = a.crow[kr] + sub;
  r.e1 = a.crow[kr + 1u];  // (a row holds its diagonal at least)
#pragma unroll
  for (int q = 0; q < SPMV_AHEAD; ++q) {
    const uint32_t e = min(r.e0 + q * SPMV_LANES, r.e1 - 1u);
    c[q] = a.ccol[e];
    r.v[q] = a.cval[e];
  }
  r.own = a.zp[kr];
#pragma unroll
  for (int q = 0; q < SPMV_AHEAD; ++q) r.w[q] = a.zp[c[q]];
}

// Writes p and q of the row; returns the lane's share of p.q.
__device__ __forceinline__ double spmv_row(const CgArgs& a, uint32_t k, uint32_t sub, double beta, const SpmvRow& r) {
  double s = 0.0;
#pragma unroll
  for (int q = 0; q < SPMV_AHEAD; ++q)
    if (r.e0 + q * SPMV_LANES < r.e1) s += r.v[q] * (r.w[q].x + beta * r.w[q].y);
  for (uint32_t e = r.e0 + SPMV_AHEAD * SPMV_LANES; e < r.e1; e += SPMV_LANES) {
    const double2 t = a.zp[a.ccol[e]];
    s += a.cval[e] * (t.x + beta * t.y);
  }
#pragma unroll
  for (int o = 1; o < SPMV_LANES; o <<= 1) s += __shfl_xor(s, o, WAVE);
  if (k >= a.m || sub != 0u) return 0.0;
  const double pk = r.own.x + beta * r.own.y;
  a.p[k] = pk;
  a.q[k] = s;
  return pk * s;
}

__global__ void __launch_bounds__(SPMV_NT) k_cg_spmv(CgArgs a, uint32_t it) {
  constexpr int NW = SPMV_NT / WAVE;
  __shared__ double sh[NW], sh_pq[NW];
  const uint32_t sub = threadIdx.x % SPMV_LANES;
  const uint32_t block = row_block();
  uint32_t k = block * SPMV_ROWS + threadIdx.x / SPMV_LANES;
  SpmvRow row;
  const uint32_t done = a.scal->done;
  double old = a.scal->rz[(it + 1u) & 1u];
  double share = part_share<NW>(a.part_rz, a.nb);
  spmv_fetch(a, k, sub, row);
  asm volatile("" : "+v"(old));  // (fetched here, not behind the sum)
  const double rz = block_sum<NW>(share, sh);
  if (done) return;
  const double beta = it && old != 0.0 ? rz / old : 0.0;
  if (blockIdx.x == 0 && threadIdx.x == 0) a.scal->rz[it & 1u] = rz;
  double pq = spmv_row(a, k, sub, beta, row);
  // block-uniform loop over row groups, so the sums run with every lane
  for (uint32_t k0 = (block + gridDim.x) * SPMV_ROWS; k0 < a.m; k0 += gridDim.x * SPMV_ROWS) {
    k += gridDim.x * SPMV_ROWS;
    spmv_fetch(a, k, sub, row);
    pq += spmv_row(a, k, sub, beta, row);
  }
  const double t = block_sum<NW>(pq, sh_pq);
  if (threadIdx.x == 0) a.part_pq[block] = t;
}

// x += alpha p, r -= alpha q, (z, p) = (D^-1 r, p); partials of r.z and r.r.
__global__ void __launch_bounds__(NT) k_cg_update(CgArgs a, uint32_t it) {
  __shared__ double sh[NT / WAVE];
  __shared__ double2 sh2[NT / WAVE];
  const uint32_t block = row_block();
  uint32_t k = block * NT + threadIdx.x;
  // the first elements are on their way while alpha is summed
  const uint32_t kr = min(k, a.m - 1u);
  const uint32_t done = a.scal->done;
  double rz0 = a.scal->rz[it & 1u];
  double pk = a.p[kr], qk = a.q[kr], xk = a.x[kr], r0 = a.r[kr], dk = a.dinv[kr];
  double share = part_share(a.part_pq, a.ns);
  asm volatile("" : "+v"(rz0));  // (fetched here, not behind the sum)
  const double pq = block_sum(share, sh);
  if (done) return;
  const double alpha = pq != 0.0 ? rz0 / pq : 0.0;
  double rz = 0.0, rr = 0.0;
  while (k < a.m) {
    a.x[k] = xk + alpha * pk;
    const double rk = r0 - alpha * qk;
    const double zk = dk * rk;
    a.r[k] = rk;
    a.zp[k] = make_double2(zk, pk);
    rz += rk * zk;
    rr += rk * rk;
    k += gridDim.x * NT;
    if (k < a.m) {
      pk = a.p[k];
      qk = a.q[k];
      xk = a.x[k];
      r0 = a.r[k];
      dk = a.dinv[k];
    }
  }
  const double2 t = block_sum2(rz, rr, sh2);
  if (threadIdx.x == 0) {
    a.part_rz[block] = t.x;
    a.part_rr[block] = t.y;
  }
}

// One block: relative residual after `it` iterations.  From convergence on
// (or a residual that is no number) the queued iterations do nothing.
__global__ void __launch_bounds__(NT) k_cg_check(CgArgs a, uint32_t it, double tol, CgScal* host) {
  __shared__ double sh[NT / WAVE];
  CgScal* sc = a.scal;
  if (it == 0 || !sc->done) {
    const double rr = block_sum(part_share(a.part_rr, a.nb), sh);
    if (threadIdx.x != 0) return;
    const double bb = it ? sc->bb : rr;
    // (a sum that is no number stays one: it compares false with zero)
    const double res = bb > 0.0 ? sqrt_cr((rr < 0.0 ? 0.0 : rr) / bb) : 0.0;
    sc->bb = bb;
    sc->res = res;
    sc->done = res <= tol ? CG_CONVERGED : (res < __longlong_as_double(0x7FF0000000000000ll) ? 0u : CG_BROKEN);
  }
  if (threadIdx.x == 0) *host = *sc;
}

// One block: source and sink currents.
__global__ void __launch_bounds__(NT) k_cg_currents(CgArgs a, CgScal* host) {
  __shared__ double2 sh[NT / WAVE];
  const double2 t = block_sum2(part_share(a.part_rz, a.nb), part_share(a.part_rr, a.nb), sh);
  if (threadIdx.x != 0) return;
  CgScal c = *a.scal;
  c.isrc = t.x;
  c.isnk = t.y;
  *host = c;
}

// Partials of the source current sum bs (1 - x) and the sink current sum bk x.
__global__ void __launch_bounds__(NT) k_cg_current(uint32_t m, const double* __restrict__ bs,
                                                   const double* __restrict__ bk,
                                                   const double* __restrict__ x,
                                                   double* __restrict__ part) {
  __shared__ double2 sh[NT / WAVE];
  double is = 0.0, ik = 0.0;
  for (uint32_t k = blockIdx.x * NT + threadIdx.x; k < m; k += gridDim.x * NT) {
    is += bs[k] * (1.0 - x[k]);
    ik += bk[k] * x[k];
  }
  const double2 t = block_sum2(is, ik, sh);
  if (threadIdx.x == 0) {
    part[blockIdx.x] = t.x;
    part[CG_MAX_BLOCKS + blockIdx.x] = t.y;
  }
}

// Potentials of every rod: solved, electrode potential, or NaN (floating).
__global__ void __launch_bounds__(NT) k_cs_potential(uint32_t n, const uint32_t* __restrict__ labels,
                                                     const uint32_t* __restrict__ flag,
                                                     const uint32_t* __restrict__ act,
                                                     const uint32_t* __restrict__ idx,
                                                     const double* __restrict__ x,
                                                     double* __restrict__ v) {
  for (uint32_t i = blockIdx.x * NT + threadIdx.x; i < n; i += gridDim.x * NT) {
    const uint32_t f = flag[labels[i]];
    double vi = __longlong_as_double(0x7FF8000000000000ll);
    if (act[i])
      vi = x[idx[i]];
    else if (f == 1u)
      vi = 1.0;
    else if (f == 2u)
      vi = 0.0;
    v[i] = vi;
  }
}

int grid_for(uint64_t n, int cap) {
  uint64_t b = (n + NT - 1) / NT;
  if (b > (uint64_t)cap) b = cap;
  if (b < 1) b = 1;
  return (int)b;
}

}  // namespace

void cg_grids(CgArgs& a) {
  auto grid = [&](uint32_t per) { return std::min<uint32_t>((a.m + per - 1u) / per, CG_MAX_BLOCKS); };
  a.nb = grid(NT);
  a.ns = grid(SPMV_ROWS);
}

void launch_cs_flag(const uint32_t* nrow, const uint32_t* ncol, const uint32_t* labels, uint32_t n,
                    uint32_t* flag, hipStream_t s) {
  hipLaunchKernelGGL(k_cs_flag, dim3(64), dim3(NT), 0, s, nrow, ncol, labels, n, flag);
}

void launch_cs_active(const uint32_t* nrow, const uint32_t* ncol, const uint32_t* labels,
                      const uint32_t* flag, uint32_t n, uint32_t* act, uint32_t* rl, hipStream_t s) {
  hipLaunchKernelGGL(k_cs_active, dim3(grid_for(n, 8192)), dim3(NT), 0, s, nrow, ncol, labels, flag,
                     n, act, rl);
}

void launch_cs_fill(const uint32_t* nrow, const uint32_t* ncol, const double* nval, uint32_t n,
                    const uint32_t* act, const uint32_t* idx, const uint32_t* off, uint32_t* crow,
                    uint32_t* ccol, double* cval, double* dinv, double* bsrc, double* bsnk,
                    hipStream_t s) {
  hipLaunchKernelGGL(k_cs_fill, dim3(grid_for(n, 8192)), dim3(NT), 0, s, nrow, ncol, nval, n, act,
                     idx, off, crow, ccol, cval, dinv, bsrc, bsnk);
}

void launch_cs_potential(uint32_t n, const uint32_t* labels, const uint32_t* flag,
                         const uint32_t* act, const uint32_t* idx, const double* x, double* v,
                         hipStream_t s) {
  hipLaunchKernelGGL(k_cs_potential, dim3(grid_for(n, 8192)), dim3(NT), 0, s, n, labels, flag, act,
                     idx, x, v);
}

void launch_cs_order(uint32_t n, const uint32_t* ord, const uint32_t* act, const uint32_t* rl, uint32_t* acto,
                     uint32_t* rlo, const uint32_t* idxo, const uint32_t* offo, uint32_t* idx, uint32_t* off,
                     int stage, hipStream_t s) {
  if (stage == 0)
    hipLaunchKernelGGL(k_cs_to_order, dim3(grid_for(n, 8192)), dim3(NT), 0, s, n, ord, act, rl, acto, rlo);
  else
    hipLaunchKernelGGL(k_cs_from_order, dim3(grid_for((uint64_t)n + 1, 8192)), dim3(NT), 0, s, n, ord, idxo, offo,
                       idx, off);
}

void launch_cg_init(const CgArgs& a, double tol, CgScal* host, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_init, dim3(a.nb), dim3(NT), 0, s, a);
  hipLaunchKernelGGL(k_cg_check, dim3(1), dim3(NT), 0, s, a, 0u, tol, host);
}

void launch_cg_iterations(const CgArgs& a, uint32_t it, uint32_t count, double tol, CgScal* host, hipStream_t s) {
  for (uint32_t j = it; j < it + count; ++j) {
    hipLaunchKernelGGL(k_cg_spmv, dim3(a.ns), dim3(SPMV_NT), 0, s, a, j);
    hipLaunchKernelGGL(k_cg_update, dim3(a.nb), dim3(NT), 0, s, a, j);
  }
  hipLaunchKernelGGL(k_cg_check, dim3(1), dim3(NT), 0, s, a, it + count, tol, host);
}

void launch_cg_current(const CgArgs& a, CgScal* host, hipStream_t s) {
  hipLaunchKernelGGL(k_cg_current, dim3(a.nb), dim3(NT), 0, s, a.m, a.bsrc, a.bsnk, a.x, a.part_rz);
  hipLaunchKernelGGL(k_cg_currents, dim3(1), dim3(NT), 0, s, a, host);
}

}  // namespace nf
