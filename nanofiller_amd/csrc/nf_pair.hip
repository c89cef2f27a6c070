// nf_pair.hip - the cell-pair engine.
//
// One 64-lane wavefront (one workgroup) per work item, a home cell or a part
// of one (k_items), taken from 64 work queues (eight per XCD, each counter on
// its own cache line).  The home
// cell's probes are taken 64 at a time, one per lane, and read by the
// other lanes with readlane.  The stencil, sorted by minimum cell-to-cell
// distance, is looked up 64 offsets at a time (one round trip), and the
// neighbour cells that can reach the chunk are packed into a 128-slot
// staging buffer (two slots per lane).  Every (probe, slot) pair passes a
// conservative filter; survivors queue in LDS, go
// through the rigorous FP32 screen 64 at a time, and those the screen
// cannot settle get the full FP32-band / FP64 test 64 at a time, so each
// expensive step runs on dense work.
//
// Modes replace the reference's kernels:
//   PM_GEN_OLD    new vs accepted rods   cuda_OldExtIsectLB (inc/intersection_kern.h:245-364)
//                 (run accepted-major, with the roles of the two sets
//                 swapped, once an instance's accepted rods outnumber the
//                 round's proposals four to one; otherwise a cut proposal
//                 leaves its stencil walk)
//   PM_GEN_NEW    new vs new, priority   cuda_InternalIsect_noLck / cuda_NewExtIsectLB_parted
//                                        (inc/intersection_kern.h:12-241)
//                 (over the first pass's survivors, compacted per cell;
//                 half stencil: each pair of them once; a cut clears the
//                 later slot's survivor flag)
//   PM_CNT        contact records        core_cell_interact_kernel CONTACT_COUNT and
//                                        CONTACT_RECORD in one pass (appended, unsorted)
//                                        (src/core_cell_interaction_kernel.cu:70-315)
#include "nf_internal.h"
#include "nf_line.h"

namespace nf {

constexpr int PAIR_THREADS = WAVE;

// Largest of the lanes' values, which are not negative, in every lane (uniform).
// Without shuffles: their lane addresses, six registers that live through the
// kernel, had been spilled and fetched again for every cell.
__device__ __forceinline__ float wave_max(float v) {
  auto step = [&](int w) { v = fmaxf(v, __int_as_float(w)); };
#define NF_DPP(CTRL, ROWS) __builtin_amdgcn_update_dpp(0, __float_as_int(v), CTRL, ROWS, 0xF, false)
  step(NF_DPP(0xB1, 0xF));   // lane ^ 1
  step(NF_DPP(0x4E, 0xF));   // lane ^ 2
  step(NF_DPP(0x141, 0xF));  // the other quad of eight lanes
  step(NF_DPP(0x140, 0xF));  // the other eight of a row of 16
  step(NF_DPP(0x142, 0xA));  // row before, into rows 1 and 3
  step(NF_DPP(0x143, 0xC));  // rows 0 and 1, into rows 2 and 3
#undef NF_DPP
  return __int_as_float(__builtin_amdgcn_readlane(__float_as_int(v), 63));
}

__device__ __forceinline__ uint32_t wave_sum(uint32_t v) {
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v += __shfl_xor(v, o, WAVE);
  return v;
}

__device__ __forceinline__ int32_t pack_img(int x, int y, int z) {
  return (int32_t)(((uint32_t)(x & 0xFF)) | ((uint32_t)(y & 0xFF) << 8) |
                   ((uint32_t)(z & 0xFF) << 16));
}

struct CellGeom {
  double box[3];
  float boxf[3];
  int nc[3];
  float rnc[3];  // 1 / nc (rounded): periodic wrap without integer division
  uint32_t cell_base;
  const int4* st;
  uint32_t st_n;
  float ew, hl_max, R_max;
  float edge[3];
  double sf64, sep64;
  float sf32, sep32;
  uint32_t cap;
  InstState* state;
  // home and neighbour rod sets of the pass; the reject-vs-accepted pass of
  // an instance whose accepted rods outnumber its proposals runs
  // accepted-major (inv): accepted rods are the probes, proposals the
  // staged neighbours, and a cut clears the proposal's alive flag directly
  const float4* hP;
  const float4* hD;
  const uint32_t* hX;
  const uint32_t* hStart;
  const uint32_t* hCount;
  const float4* nP;
  const float4* nD;
  const uint32_t* nX;
  const uint32_t* nStart;
  const uint32_t* nCount;
  const float* nHl;
  bool inv;
  bool idle;  // reject-vs-accepted pass: the instance has no proposals, or no accepted rods
};

// Per-lane statistics, flushed to the instance (or the contact counters)
// by every lane together; lanes other than 0 add zero.
struct Acc {
  uint32_t tests, rech, kills;
  double maxdd;
  unsigned long long bytes;  // wave-uniform: probe and tile bytes streamed
};

// Values the hardware must treat as wave-uniform: read from lane 0 into an
// SGPR so that every branch and loop bound that depends on them is scalar.
// The pair engine keeps all control flow outside the innermost tile loop
// uniform in this way, and performs cross-lane operations (shuffles,
// ballots, barriers) only where every lane of the wave is active.
__device__ __forceinline__ uint32_t uni(uint32_t v) {
  return (uint32_t)__builtin_amdgcn_readfirstlane((int)v);
}
__device__ __forceinline__ int unii(int v) { return __builtin_amdgcn_readfirstlane(v); }
__device__ __forceinline__ float unif(float v) {
  return __int_as_float(__builtin_amdgcn_readfirstlane(__float_as_int(v)));
}

template <bool GEN>
__device__ __forceinline__ void flush(const PairArgs& a, const CellGeom& g, Acc& acc, int mode) {
  const uint32_t wt = wave_sum(acc.tests), wr = wave_sum(acc.rech), wk = wave_sum(acc.kills);
  double v = acc.maxdd;
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, WAVE));
  const bool l0 = threadIdx.x == 0;
  unsigned long long* c0;
  unsigned long long* c1;
  unsigned long long* c2;
  unsigned long long* c3;
  if (GEN) {
    c0 = &g.state->pair_tests;
    c1 = &g.state->rechecks;
    c2 = &g.state->rej_new;
    c3 = (unsigned long long*)&g.state->max_dd;
  } else {
    c0 = &a.ctr[0];
    c1 = &a.ctr[1];
    c2 = &a.ctr[3];  // unused for contacts
    c3 = &a.ctr[2];
  }
  // lane 0 alone issues the atomics: nothing in this branch is cross-lane,
  // and the caller's next cross-lane operation follows the reconvergence
  unsigned long long* cb =
      GEN ? (mode == PM_GEN_OLD ? &g.state->tile_bytes : &g.state->tile_bytes_new) : &a.ctr[3];
  if (l0) {
    atomicAdd(c0, (unsigned long long)wt);
    atomicAdd(c1, (unsigned long long)wr);
    // rejections by earlier proposals of the round (the round controller
    // counts those by accepted rods from the survivor counts)
    if (GEN && mode == PM_GEN_NEW) atomicAdd(c2, (unsigned long long)wk);
    atomicMax(c3, (unsigned long long)__double_as_longlong(v));
    atomicAdd(cb, acc.bytes);
  }
  acc.tests = acc.rech = acc.kills = 0;
  acc.maxdd = 0.0;
  acc.bytes = 0;
}

// LDS of one wave (under 10 KB, so 16 waves fit a CU): the probe chunk, the
// staged neighbour rods and the two pair queues.  The probes still in the
// walk sit at the front, in lane order (compact_probes).
constexpr int SLOTS = 2 * WAVE;
constexpr int QCAP = 2 * WAVE;   // fewer than 64 wait between pushes of up to 64
constexpr int PUNROLL = 4;       // probes per trip of the filter loop
struct PairLds {
  float4 sP[WAVE], sD[WAVE];  // probes of the chunk
  float4 pf[WAVE];            // filter: direction, x of the moment (every pair: 2 (P - o), 2 rp)
  float2 pg[WAVE];            // filter: y and z of the moment (every pair: |P - o|^2 - rp^2 - slack)
  uint32_t sX[WAVE];
  uint32_t hit[WAVE];           // per probe: overlaps something (generation)
  float4 bP[SLOTS], bD[SLOTS];  // staged neighbour rods
  uint32_t bX[SLOTS];           // rod id (0xFFFFFFFF: not a candidate)
  uint32_t bM[SLOTS];           // image code | same cell << 31
  uint32_t qE[QCAP];            // queued pairs: probe | slot << 8
  uint32_t q2[QCAP];            // pairs for the full test: probe | slot << 8 | fp64 << 16
};

__device__ __forceinline__ uint32_t lane_prefix(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32),
                                   __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ int img_x(uint32_t meta) { return (int)(int8_t)(meta & 0xFF); }
__device__ __forceinline__ int img_y(uint32_t meta) { return (int)(int8_t)((meta >> 8) & 0xFF); }
__device__ __forceinline__ int img_z(uint32_t meta) { return (int)(int8_t)((meta >> 16) & 0xFF); }

// FP32 image shift of a neighbour: the FP64 shift img * box rounded once.
// Box edges are float-exact (nf_params_normalize) and |img| < 128, so the
// product is exact in FP64 and the FP32 product rounds the same exact value
// once: (float)img * boxf is that rounding, without FP64 arithmetic.
__device__ __forceinline__ float3 shift_f32(const CellGeom& g, uint32_t meta) {
  return make_float3((float)img_x(meta) * g.boxf[0], (float)img_y(meta) * g.boxf[1],
                     (float)img_z(meta) * g.boxf[2]);
}

// Screen of one queued pair (valid lanes only): the reach band and the
// line-distance bound of pair_f32_screen.  Counts the pair test when reach
// is decided.  Returns 0 (settled), 1 (full FP32 test needed) or 2 (reach
// undecided, or the plain FP64 path: the full test decides reach and cut in
// FP64 and counts).
template <int MODE, int PREC>
__device__ __forceinline__ uint32_t screen_test(const PairArgs& a, const CellGeom& g, PairLds& L,
                                                uint32_t e, bool valid, Acc& acc) {
  constexpr bool GEN = (MODE == PM_GEN_OLD || MODE == PM_GEN_NEW);
  const uint32_t ent = L.qE[e];
  const uint32_t p = ent & 0xFFu, j = ent >> 8;
  if (PREC == NF_PREC_FP64) return valid ? 2u : 0u;
  const float4 P2 = L.bP[j], D2 = L.bD[j];
  const uint32_t meta = L.bM[j];
  const float4 P1 = L.sP[p], D1 = L.sD[p];
  if (!valid) return 0u;
  const float3 sh = shift_f32(g, meta);
  const float R32 = GEN ? (g.sf32 * (D1.w + D2.w) + g.sep32) : ((D1.w + D2.w) + a.gap32);
  const int r = pair_f32_screen(P1, D1, P2, D2, sh.x, sh.y, sh.z, R32, g.ew);
  if (r == SCREEN_UNDECIDED) return 2u;
  if (r == SCREEN_OUT) return 0u;
  ++acc.tests;
  return r == SCREEN_FULL ? 1u : 0u;
}

// Full capsule test of one pair of the second queue (valid lanes only): the
// FP32 band with FP64 recheck, or plain FP64 (flag bit 16: reach not yet
// decided, count here).  No cross-lane operation inside.
template <int MODE, int PREC>
__device__ __forceinline__ void full_test(const PairArgs& a, const CellGeom& g, PairLds& L,
                                          uint32_t e, bool valid, Acc& acc) {
  constexpr bool GEN = (MODE == PM_GEN_OLD || MODE == PM_GEN_NEW);
  const uint32_t ent = L.q2[e];
  const uint32_t p = ent & 0xFFu, j = (ent >> 8) & 0xFFu;
  const bool f64 = PREC == NF_PREC_FP64 || ((ent >> 16) & 1u) != 0u;
  const float4 P2 = L.bP[j], D2 = L.bD[j];
  const uint32_t meta = L.bM[j];
  const uint32_t xj = L.bX[j];
  const float4 P1 = L.sP[p], D1 = L.sD[p];
  const uint32_t X1 = L.sX[p];
  if (!valid) return;
  const int ix = img_x(meta), iy = img_y(meta), iz = img_z(meta);
  const double sx = (double)ix * g.box[0], sy = (double)iy * g.box[1], sz = (double)iz * g.box[2];
  // FP64 evaluation in the canonical orientation the decisions are defined
  // by: generation puts the probe (proposal, or the later slot) first;
  // contacts put the lower rod id first, with the periodic image applied to
  // the higher id.  The closest-point solve is not bitwise symmetric under
  // swapping the segments.
  // generation: the later slot first (same-round pass), the proposal first
  // (reject-vs-accepted, swapped when run accepted-major)
  const bool swap = MODE == PM_GEN_NEW ? (X1 < xj) : (GEN ? g.inv : (X1 > xj));
  const float4 Pa = swap ? P2 : P1, Da = swap ? D2 : D1;
  const float4 Pb = swap ? P1 : P2, Db = swap ? D1 : D2;
  const double ux = swap ? -sx : sx, uy = swap ? -sy : sy, uz = swap ? -sz : sz;
  bool within = true;
  bool cut;
  double d2_64 = -1.0;
  double R64;
  if (GEN)
    R64 = g.sf64 * ((double)D1.w + (double)D2.w) + g.sep64;
  else
    R64 = ((double)Da.w + (double)Db.w) + a.gap64;
  if (f64) {
    if (PREC != NF_PREC_FP64) ++acc.rech;
    d2_64 = pair_d2_f64(Pa, Da, Pb, Db, ux, uy, uz, R64, &within);
    cut = GEN ? (d2_64 < R64 * R64) : (d2_64 <= R64 * R64);
    if (!within) return;
    ++acc.tests;
  } else {
    // reach was decided 'within' by the screen with the same band
    const float R32 = GEN ? (g.sf32 * (D1.w + D2.w) + g.sep32) : ((D1.w + D2.w) + a.gap32);
    const F32Pair r = pair_f32(P1, D1, P2, D2, (float)sx, (float)sy, (float)sz, R32, g.ew, GEN);
    if (r.decided < 0) {
      ++acc.rech;
      bool w64;
      d2_64 = pair_d2_f64(Pa, Da, Pb, Db, ux, uy, uz, R64, &w64);
      cut = GEN ? (d2_64 < R64 * R64) : (d2_64 <= R64 * R64);
    } else {
      cut = r.decided != 0;
      if (a.diag) {
        bool w2;
        const double e64 = pair_d2_f64(Pa, Da, Pb, Db, ux, uy, uz, R64, &w2);
        const double dd = fabs(sqrt((double)r.d2) - sqrt(e64));
        acc.maxdd = dd > acc.maxdd ? dd : acc.maxdd;
      }
    }
  }
  if (!cut) return;
  if (MODE == PM_GEN_NEW) {
    // the later slot loses; several earlier ones may cut it, count it once
    const uint32_t loser = X1 > xj ? X1 : xj;
    if (atomicExch(&a.surv[loser], 0u) != 0u) ++acc.kills;
  } else if (GEN) {
    if (g.inv)
      a.alive_out[xj] = 0u;  // accepted-major: the slot is the proposal (xj its index)
    else
      L.hit[p] = 1u;
  } else {
    if (d2_64 < 0.0) {
      bool w2;
      d2_64 = pair_d2_f64(Pa, Da, Pb, Db, ux, uy, uz, R64, &w2);
    }
    // append to the unsorted list; the host sizes the buffer again and
    // repeats the pass when the count exceeds its capacity
    const uint32_t I = X1 < xj ? X1 : xj;
    const uint32_t J = X1 < xj ? xj : X1;
    const int sgn = X1 < xj ? 1 : -1;
    const uint32_t pos = atomicAdd(a.app_n, 1u);
    if (pos >= a.app_cap) return;
    const double gv = sqrt_cr(d2_64) - ((double)Da.w + (double)Db.w);
    a.outI[pos] = I;
    a.outJ[pos] = J;
    a.outGap[pos] = (float)gv;
    a.outGap64[pos] = gv;
    a.outImg[pos] = pack_img(sgn * ix, sgn * iy, sgn * iz);
  }
}

// Moves entries [base, base + cnt) of the first queue through the screen
// and appends those that need the full test to the second queue; runs the
// full test when 64 are waiting.  Wave-uniform control; the caller holds a
// barrier before the call.
template <int MODE, int PREC>
__device__ __forceinline__ void screen_batch(const PairArgs& a, const CellGeom& g, PairLds& L,
                                             uint32_t base, uint32_t cnt, uint32_t& q2n,
                                             Acc& acc) {
  const int lane = threadIdx.x;
  const bool valid = (uint32_t)lane < cnt;
  const uint32_t e = base + min((uint32_t)lane, cnt - 1u);
  const uint32_t code = screen_test<MODE, PREC>(a, g, L, e, valid, acc);
  const bool f = code != 0u;
  const unsigned long long mask = __ballot(f);
  if (f) L.q2[q2n + lane_prefix(mask)] = L.qE[e] | (code == 2u ? 0x10000u : 0u);
  q2n += (uint32_t)__popcll(mask);
  if (q2n >= (uint32_t)WAVE) {
    __syncthreads();
    full_test<MODE, PREC>(a, g, L, q2n - WAVE + (uint32_t)lane, true, acc);
    q2n -= WAVE;
  }
  __syncthreads();
}

// Walk state over the sorted stencil of one probe chunk.  The stencil is
// taken 64 offsets at a time: every lane looks up one neighbour cell (count,
// start and longest rod in parallel, one round trip) and keeps it in
// registers (cS, cN, cM); the relevant ones form a wave-uniform lane mask,
// taken in stencil (lane) order with readlane.  All other fields are
// wave-uniform.
struct StencilCursor {
  uint32_t sb;              // next stencil block (first offset of this work item)
  uint32_t nst;             // stencil parts of the cell: the item's offsets lie nst apart
  unsigned long long mask;  // relevant cells of the block not yet taken
  uint32_t cS, cN, cM;      // per lane: the lane's cell of the block
  uint32_t start;           // current neighbour cell: first index, rod count, staged so far
  uint32_t n;
  uint32_t off;
  uint32_t meta;            // image code | same cell << 31
  bool last;                // no stencil block left after the current one
  bool done;
};

template <int MODE>
__device__ void refill_cells(const PairArgs& a, const CellGeom& g, PairLds& L, StencilCursor& c,
                             int c0, int c1, int c2, float chunk_hl, float rr_chunk2) {
  const int lane = threadIdx.x;
  while (!c.last) {
    const uint32_t si = c.sb + (uint32_t)lane * c.nst;
    const bool valid = si < g.st_n;
    const int4 so = g.st[min(si, g.st_n - 1u)];
    const float md2 = __int_as_float(so.w);
    const int raw[3] = {c0 + so.x, c1 + so.y, c2 + so.z};
    int img[3], m[3];
    // image = floor(raw / nc): the float quotient of raw + 1/2 is at least
    // 1/(2 nc) from an integer and its rounding error is far below that for
    // |raw| < 2^21, so the floor is exact (checked against integer division
    // for every nc <= 1024)
#pragma unroll
    for (int d = 0; d < 3; ++d) {
      const int q = (int)floorf(((float)raw[d] + 0.5f) * g.rnc[d]);
      img[d] = q;
      m[d] = raw[d] - q * g.nc[d];
    }
    const uint32_t nc = g.cell_base + (uint32_t)(m[0] + g.nc[0] * (m[1] + g.nc[1] * m[2]));
    uint32_t n = g.nCount[nc];
    const float hl = g.nHl[nc];
    const uint32_t st0 = g.nStart[nc];
    // the three loads in flight together: the compiler would otherwise sink
    // the second behind a branch on the count and the third past the loop,
    // three dependent round trips instead of one
    asm volatile("" ::"v"(n), "v"(hl), "v"(st0));
    if (MODE == PM_GEN_OLD && !g.inv) n = min(n, g.cap);  // accepted cells hold at most cap rods
    const float rr_c = (chunk_hl + hl) * 1.000001f + g.R_max + CELL_MARGIN;
    const bool beyond = valid && md2 > rr_chunk2;
    const bool rel = valid && !beyond && n > 0u && md2 <= rr_c * rr_c;
    const unsigned long long mk = __ballot(rel);
    const bool same = so.x == 0 && so.y == 0 && so.z == 0;
    c.cS = st0;
    c.cN = n;
    c.cM = (uint32_t)pack_img(img[0], img[1], img[2]) | (same ? 0x80000000u : 0u);
    const bool stop = (__ballot(beyond) != 0ull) || (c.sb + WAVE * c.nst >= g.st_n);
    c.sb += WAVE * c.nst;
    c.mask = mk;
    if (stop) c.last = true;
    if (mk != 0ull) return;
  }
}

// Advances to the next relevant neighbour cell (stencil sorted by minimum
// cell distance: the first block with an offset past the chunk's reach is
// the last one).
template <int MODE>
__device__ __forceinline__ void next_cell(const PairArgs& a, const CellGeom& g, PairLds& L,
                                          StencilCursor& c, int c0, int c1, int c2,
                                          float chunk_hl, float rr_chunk2) {
  if (c.mask == 0ull) {
    if (!c.last) refill_cells<MODE>(a, g, L, c, c0, c1, c2, chunk_hl, rr_chunk2);
    if (c.mask == 0ull) {
      c.done = true;
      return;
    }
  }
  const int i = (int)__builtin_ctzll(c.mask);
  c.mask &= c.mask - 1ull;
  c.start = (uint32_t)__builtin_amdgcn_readlane((int)c.cS, i);
  c.n = (uint32_t)__builtin_amdgcn_readlane((int)c.cN, i);
  c.meta = (uint32_t)__builtin_amdgcn_readlane((int)c.cM, i);
  c.off = 0u;
}

// Constants of the filter for one home cell.
struct Filter {
  float3 o;       // origin: the cell's centre
  LineFilter ln;  // nf_line.h (every pair: slack 64 u S^2, see process_cell)
};

// Shifts a pair's verdict into the word: 1 when the lines may come within the
// cut distance, or (every pair) the centres within reach.
template <bool ALL>
__device__ __forceinline__ uint32_t may_cut(const float4 f, const float2 h, const SlotSide& q, uint32_t word) {
  return __builtin_amdgcn_alignbit(word, __float_as_uint(slot_apart<ALL>(f, h, q)), 31u);
}

template <bool ALL>
__device__ __forceinline__ SlotSide slot_pre(const float4 P, const float4 D, const float3 sh, const Filter& F,
                                             bool valid) {
  return slot_side<ALL>(F.ln, (P.x + sh.x) - F.o.x, (P.y + sh.y) - F.o.y, (P.z + sh.z) - F.o.z, P.w, D, valid);
}

// Appends the pairs of a word of probes per slot of the lane (bit k: probe base
// + k; m1: the second slot) to the first queue, screening 64 at a time when
// enough wait.
template <int MODE, int PREC, bool TWO>
__device__ __forceinline__ void push_pairs(const PairArgs& a, const CellGeom& g, PairLds& L, uint32_t m0, uint32_t m1,
                                           uint32_t base, uint32_t& qn, uint32_t& q2n, Acc& acc) {
  const uint32_t lane = threadIdx.x;
  for (;;) {
    const bool f0 = m0 != 0u, f = TWO ? (m0 | m1) != 0u : f0;
    const unsigned long long m = __ballot(f);
    if (m == 0ull) return;
    const uint32_t w = TWO && !f0 ? m1 : m0;
    const uint32_t k = base + (uint32_t)__builtin_ctz(w | 0x80000000u);
    const uint32_t code = k | ((TWO && !f0 ? lane + (uint32_t)WAVE : lane) << 8);
    if (TWO && !f0)
      m1 &= m1 - 1u;
    else
      m0 &= m0 - 1u;
    if (f) L.qE[qn + lane_prefix(m)] = code;
    qn += (uint32_t)__popcll(m);
    if (qn >= (uint32_t)WAVE) {
      __syncthreads();
      screen_batch<MODE, PREC>(a, g, L, qn - WAVE, WAVE, q2n, acc);
      qn -= WAVE;
    }
  }
}

// Filter of every (probe, slot) pair of one staged batch, the lanes spanning
// the slots (one each, or two when the batch fills the second half), the
// probes read from LDS by all lanes at once.  A lane gathers the verdicts of
// 32 probes in one word per slot and only then turns to the pairs that
// passed, so the loop is 12 VALU instructions per 64 pairs (6 with the centre
// filter of ALL) without a branch, ballot or queue write.  keep0, keep1: the
// pairs that the pass's ordering allows (half-stencil passes).
template <int MODE, int PREC, bool ALL, bool TWO>
__device__ __forceinline__ void probe_loop(const PairArgs& a, const CellGeom& g, PairLds& L, uint32_t nprobe,
                                           const SlotSide& Q0, const SlotSide& Q1, unsigned long long keep0,
                                           unsigned long long keep1, uint32_t& qn, uint32_t& q2n, Acc& acc) {
  constexpr bool ORD = (MODE == PM_CNT || MODE == PM_GEN_NEW);
  for (uint32_t w = 0; w < nprobe; w += 32u) {
    uint32_t m0 = 0u, m1 = 0u;
    // the first probe ends in bit 0
    const uint32_t n = min(32u, nprobe - w);
    int k = (int)((n + PUNROLL - 1u) & ~(uint32_t)(PUNROLL - 1));
    while (k > 0) {
      k -= PUNROLL;
      const uint32_t at = w + (uint32_t)k;
#pragma unroll
      for (int u = PUNROLL - 1; u >= 0; --u) {
        const float4 f = L.pf[at + (uint32_t)u];
        const float2 h = L.pg[at + (uint32_t)u];
        m0 = may_cut<ALL>(f, h, Q0, m0);
        if (TWO) m1 = may_cut<ALL>(f, h, Q1, m1);
      }
    }
    const uint32_t some = n < 32u ? (1u << n) - 1u : ~0u;  // the rows past the last probe
    m0 &= some;
    m1 &= some;
    if (ORD) {
      m0 &= (uint32_t)(keep0 >> w);
      m1 &= (uint32_t)(keep1 >> w);
    }
    push_pairs<MODE, PREC, TWO>(a, g, L, m0, m1, w, qn, q2n, acc);
  }
}

// Writes the probes of the mask (one per lane) to the front of the chunk's
// LDS tables, in lane order.  Returns the lane's place among them.
template <bool ALL>
__device__ __forceinline__ uint32_t compact_probes(const CellGeom& g, PairLds& L, unsigned long long pmask,
                                                   const float4 P1, const float4 D1, uint32_t X1, const Filter& F) {
  const uint32_t lane = threadIdx.x;
  const uint32_t at = lane_prefix(pmask);
  if ((pmask >> lane) & 1ull) {
    const float x = P1.x - F.o.x, y = P1.y - F.o.y, z = P1.z - F.o.z;
    L.sP[at] = P1;
    L.sD[at] = D1;
    L.sX[at] = X1;
    L.hit[at] = 0u;
    if (ALL) {
      const float rp = (P1.w * 1.000001f + (g.R_max + 16.0f * g.ew)) * 1.000006f;
      L.pf[at] = make_float4(2.0f * x, 2.0f * y, 2.0f * z, 2.0f * rp);
      L.pg[at] = make_float2(fmaf(z, z, fmaf(y, y, x * x)) - fmaf(rp, rp, F.ln.slack), 0.0f);
    } else {
      const LineSide l = line_side(F.ln, x, y, z, D1);
      L.pf[at] = make_float4(l.ux, l.uy, l.uz, l.mx);
      L.pg[at] = make_float2(l.my, l.mz);
    }
  }
  return at;
}

// The pairs that the ordering of a half-stencil pass keeps for one slot, bit
// k the probe of index lo + k: of the home cell's rods only the later ones of
// a probe, elsewhere (an image may map back to the home cell) never the probe
// itself.
__device__ __forceinline__ unsigned long long ordered(uint32_t src, uint32_t meta, uint32_t lo) {
  const uint32_t k = src - lo;  // wraps past 2^32 below lo
  if (meta & 0x80000000u) return src <= lo ? 0ull : (k >= 64u ? ~0ull : (1ull << k) - 1ull);
  return k >= 64u ? ~0ull : ~(1ull << k);
}

// One home cell.  For each chunk of up to 64 probes: walk the sorted
// stencil and pack the rods of consecutive relevant neighbour cells into a
// 128-slot staging buffer (two slots per lane, both loads in flight
// together, no lanes wasted on sparse cells); then run the chunk's probes
// (read by broadcast from LDS) through a conservative filter with the lanes
// spanning the slots, keep the pairs that pass in an LDS queue, screen them
// 64 at a time (reach band, line distance) and run the full test on the
// survivors 64 at a time, so every expensive step runs on dense work.
//
// What bounds the pass is VALU issue.  The filter is the distance of the two
// axes' lines (nf_line.h), which leaves about one pair in a hundred; a
// centre-distance filter leaves the fifth of the staged pairs that are within
// reach, each of which then cost some 90 instructions of gather and screen.
// Same-round pass of 4M uniform rods, MI355X: 1.65 -> 1.06 ms; 2,000 rods
// 0.10 -> 0.036 ms, 500,000 log-normal rods in agglomerates 0.49 -> 0.44 ms.
//
// Every pair within reach (ALL: the contact pass, and the generation passes
// that count pair tests as the oracle does): the full test first rejects pairs whose FP32 centre distance
// w2 exceeds rr^2 by more than its error band, rr = (hl1 + hl2) * 1.000001
// + R.  The filter keeps every pair with w2' <= rr''^2, where
// rr'' = (hl1 * 1.000001 + R_max + 16 ew) * 1.000006 + (hl2 * 1.000001) * 1.000006
// is rr' = hl1 * 1.000001 + hl2 * 1.000001 + R_max + 16 ew >= rr + 16 ew
// scaled by 1.000006 less a few float roundings (below 1e-7 relative), so
// rr''^2 >= rr'^2 * 1.00001.  The probe's part rp of rr'' is computed per
// lane, the slot's part rq is staged with the slot.  Centres are taken from
// an origin o in the home cell: p = P1 - o and q = (P2 + shift) - o are each
// within 2 ew of the exact differences, so w' = p - q differs from the full
// test's ((P1 - P2) - shift) by less than 8 ew.  The test is
//   2 p.q + 2 rp rq + (rq^2 - |q|^2) - (|p|^2 - rp^2) >= 0,
// four FMAs.  For a pair that has to pass, |q| <= |p| + rp + rq, so with
// S = |p| + rp + rq every term and partial sum is below 4 S^2; the two
// brackets take five roundings of values below S^2 each, the chain one
// subtraction and four FMAs of values below 4 S^2: 30 u S^2 in all.  The
// slack in the probe's bracket is 64 u S^2 with S bounded over the cell.
// So with ALL every pair the full test would count or cut is queued.
//
// A work item is one probe chunk group and one stencil part of a cell
// (k_items): the cell's probes are dealt into nch equal chunks of at most 64;
// the item takes the chunks cg, cg + ncg, ... and the stencil offsets sp,
// sp + nst, ..., so the ncg * nst items of a cell partition its pairs and a
// dense cell is worked on by several waves at once.  Interleaved offsets
// give every part near and far cells alike.  The probe bytes, counted per
// probe, belong to part sp = 0.
template <int MODE, int PREC, bool ALL>
__device__ void process_cell(const PairArgs& a, const CellGeom& g, uint32_t gc, uint32_t cg, uint32_t ncg,
                             uint32_t sp, uint32_t nst, PairLds& L, Acc& acc) {
  const int lane = threadIdx.x;
  // an instance without proposals (finished, or planned none) or without
  // accepted rods (its first round) has no pairs: its cells would walk their
  // stencils for nothing
  if (MODE == PM_GEN_OLD && g.idle) return;
  uint32_t pc = uni(g.hCount[gc]);
  if (MODE == PM_GEN_OLD && g.inv) pc = min(pc, g.cap);  // accepted cells hold at most cap rods
  if (pc == 0) return;
  const uint32_t nch = (pc + WAVE - 1u) / WAVE;
  const uint32_t csz = (pc + nch - 1u) / nch;  // probes per chunk
  const uint32_t ps = uni(g.hStart[gc]);
  const uint32_t lc = gc - g.cell_base;
  const int c0 = (int)(lc % (uint32_t)g.nc[0]);
  const int c1 = (int)((lc / (uint32_t)g.nc[0]) % (uint32_t)g.nc[1]);
  const int c2 = (int)(lc / ((uint32_t)g.nc[0] * (uint32_t)g.nc[1]));
  // the filter's origin (the home cell's centre), scale and slack (scalars)
  Filter F;
  F.o = make_float3(unif(((float)c0 + 0.5f) * g.edge[0]), unif(((float)c1 + 0.5f) * g.edge[1]),
                    unif(((float)c2 + 0.5f) * g.edge[2]));
  const float Smax = 0.51f * (g.edge[0] + g.edge[1] + g.edge[2]) + 2.0f * CELL_MARGIN +
                     2.00002f * (g.hl_max + g.R_max + 16.0f * g.ew);
  if (ALL)
    F.ln = LineFilter{0.0f, 64.0f * U32 * Smax * Smax};
  else
    F.ln = line_filter(g.R_max, g.ew, Smax);
  F.ln = LineFilter{unif(F.ln.scale), unif(F.ln.slack)};

  for (uint32_t pb = cg * csz; pb < pc; pb += ncg * csz) {
    const uint32_t G = min(csz, pc - pb);
    // lane l holds probe l of the chunk (clamped loads, every lane loads)
    const bool inrange = (uint32_t)lane < G;
    const uint32_t pidx = ps + pb + min((uint32_t)lane, G - 1u);
    const float4 P1 = g.hP[pidx];
    const float4 D1 = g.hD[pidx];
    const uint32_t X1 = g.hX[pidx];
    const bool have = inrange;
    // probes still in the walk, as a wave-uniform mask
    unsigned long long pmask = __ballot(have);
    const float chunk_hl = wave_max(have ? P1.w : 0.0f);
    if (sp == 0u) acc.bytes += (unsigned long long)G * 36ull;
    const float rr_chunk = (chunk_hl + g.hl_max) * 1.000001f + g.R_max + CELL_MARGIN;
    const float rr_chunk2 = rr_chunk * rr_chunk;
    uint32_t qn = 0;   // wave-uniform queue lengths: filtered pairs,
    uint32_t q2n = 0;  // and pairs waiting for the full test
    StencilCursor cur{sp, nst, 0ull, 0u, 0u, 0u, 0u, 0u, 0u, 0u, false, false};
    // several parts walk for this chunk's proposals: each tells the others of
    // its cuts through the alive flags
    const bool share = MODE == PM_GEN_OLD && !g.inv && !ALL && nst > 1u;
    uint32_t at = compact_probes<ALL>(g, L, pmask, P1, D1, X1, F);
    unsigned long long listed = pmask;  // the probes in the LDS tables
    __syncthreads();

    while (!cur.done) {
      // ---- stage: the lane's two slots take their source index from the
      // cell that covers them (registers only)
      uint32_t fill = 0;
      uint32_t src0 = 0u, src1 = 0u, m0 = 0u, m1 = 0u;
      while (fill < (uint32_t)SLOTS) {
        if (cur.off >= cur.n) {
          next_cell<MODE>(a, g, L, cur, c0, c1, c2, chunk_hl, rr_chunk2);
          if (cur.done) break;
        }
        const uint32_t take = min(cur.n - cur.off, (uint32_t)SLOTS - fill);
        const uint32_t r0 = (uint32_t)lane - fill;  // wraps past 2^32 when lane < fill
        const uint32_t r1 = (uint32_t)lane + (uint32_t)WAVE - fill;
        if (r0 < take) {
          src0 = cur.start + cur.off + r0;
          m0 = cur.meta;
        }
        if (r1 < take) {
          src1 = cur.start + cur.off + r1;
          m1 = cur.meta;
        }
        fill += take;
        cur.off += take;
      }
      if (fill == 0) break;
      acc.bytes += (unsigned long long)fill * 36ull;
      // ---- load: both slots' loads in flight together; every lane loads
      // (unfilled slots read index 0 of a non-empty array and are never used)
      const bool v0 = (uint32_t)lane < fill, v1 = (uint32_t)lane + WAVE < fill;
      const float4 p0 = g.nP[src0], p1 = g.nP[src1];
      const float4 d0 = g.nD[src0], d1 = g.nD[src1];
      // accepted-major pass: the slot keeps the proposal's index, which a
      // cut clears in the alive flags
      uint32_t x0 = src0, x1 = src1;
      if (!(MODE == PM_GEN_OLD && g.inv)) {
        x0 = g.nX[src0];
        x1 = g.nX[src1];
      }
      // the proposals that the cell's other parts have cut meanwhile
      uint32_t alive = 1u;
      if (share)
        alive = __hip_atomic_load(&a.alive_out[pidx], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      L.bP[lane] = p0;
      L.bD[lane] = d0;
      L.bX[lane] = x0;
      L.bM[lane] = m0;
      L.bP[lane + WAVE] = p1;
      L.bD[lane + WAVE] = d1;
      L.bX[lane + WAVE] = x1;
      L.bM[lane + WAVE] = m1;
      const float3 s0 = shift_f32(g, m0), s1 = shift_f32(g, m1);
      const SlotSide Q0 = slot_pre<ALL>(p0, d0, s0, F, v0), Q1 = slot_pre<ALL>(p1, d1, s1, F, v1);
      unsigned long long keep0 = ~0ull, keep1 = ~0ull;
      if (MODE == PM_CNT || MODE == PM_GEN_NEW) {
        keep0 = ordered(src0, m0, ps + pb);
        keep1 = ordered(src1, m1, ps + pb);
      }
      if (share) {
        pmask &= __ballot(alive != 0u);
        if (pmask == 0ull) break;
      }
      // probes have left the walk: the others move up
      if (MODE == PM_GEN_OLD && pmask != listed) {
        at = compact_probes<ALL>(g, L, pmask, P1, D1, X1, F);
        listed = pmask;
      }
      __syncthreads();
      // ---- filter every (probe, slot) pair, queue the survivors
      const uint32_t np = (uint32_t)__popcll(listed);
      if (fill > (uint32_t)WAVE)
        probe_loop<MODE, PREC, ALL, true>(a, g, L, np, Q0, Q1, keep0, keep1, qn, q2n, acc);
      else
        probe_loop<MODE, PREC, ALL, false>(a, g, L, np, Q0, Q1, keep0, keep1, qn, q2n, acc);
      // ---- drain both queues before the slots are restaged
      if (qn > 0) {
        __syncthreads();
        screen_batch<MODE, PREC>(a, g, L, 0u, qn, q2n, acc);
        qn = 0;
      }
      if (q2n > 0) {
        __syncthreads();
        full_test<MODE, PREC>(a, g, L, min((uint32_t)lane, q2n - 1u), (uint32_t)lane < q2n, acc);
        q2n = 0;
      }
      __syncthreads();
      if (MODE == PM_GEN_OLD && !g.inv && !ALL) {
        // a proposal once cut is rejected whatever else it overlaps: cut
        // proposals leave the walk, which ends when none is left.  The
        // stencil is sorted by distance, so near a jammed state most
        // proposals leave after their first batches.  The decisions are
        // unchanged; the pair-test count is then the pairs evaluated.
        const bool cut = ((listed >> lane) & 1ull) && L.hit[at] != 0u;
        if (cut && ((pmask >> lane) & 1ull))
          __hip_atomic_store(&a.alive_out[pidx], 0u, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
        pmask &= ~__ballot(cut);
        if (pmask == 0ull) break;
      }
    }
    // every pair tested: the cut proposals' flags now
    if (MODE == PM_GEN_OLD && !g.inv && ALL && have && L.hit[at] != 0u) a.alive_out[pidx] = 0u;
    __syncthreads();
  }
}

// Reject-vs-accepted pass: an instance's proposals of this round and accepted
// rods.  Accepted-major (inv) when the accepted rods outnumber the proposals
// four to one: fewer, denser probe chunks stage the sparser set (the pair set
// and every decision are the same).  Below that ratio the proposals are the
// probes, so that cut ones can leave their walk early.  idle: no pairs.
struct OldRoles {
  uint32_t nacc, nprop;
  bool inv, idle;
};
__device__ __forceinline__ OldRoles old_roles(const PairArgs& a, uint32_t inst, const InstDesc& d) {
  OldRoles r;
  r.nacc = a.st[inst].n_acc;
  r.nprop = a.prStart[d.cell_base + d.ncells] - a.prStart[d.cell_base];
  r.inv = r.nacc > 4u * r.nprop;
  r.idle = r.nprop == 0u || r.nacc == 0u || (a.skip_walk && d.fine.on);
  return r;
}

template <int MODE, int PREC, bool ALL>
__global__ void __launch_bounds__(PAIR_THREADS, 4) k_pair(PairArgs a) {
  __shared__ PairLds L;
  constexpr bool GEN = (MODE == PM_GEN_OLD || MODE == PM_GEN_NEW);
  const uint32_t W = a.ncells_total;
  const int xcd = blockIdx.x & 7;
  // rounds after every instance finished plan no candidates: nothing to do
  if (GEN && uni(a.ri->T) == 0u) return;
  // no instance has both candidates and accepted rods: no first-pass pairs
  if (MODE == PM_GEN_OLD && uni(a.ri->old) == 0u) return;
  const bool l0 = threadIdx.x == 0;
  CellGeom g;
  Acc acc = {0u, 0u, 0u, 0.0, 0ull};
  uint32_t cur_inst = 0xFFFFFFFFu;
  if (!GEN) {
    for (int d = 0; d < 3; ++d) {
      g.box[d] = a.box[d];
      g.boxf[d] = a.boxf[d];
      g.nc[d] = a.ncell[d];
      g.rnc[d] = 1.0f / (float)a.ncell[d];
      g.edge[d] = a.boxf[d] / (float)a.ncell[d];
    }
    g.cell_base = 0;
    g.st = a.stencil + a.st_off;
    g.st_n = a.st_n;
    g.ew = a.ew;
    g.hl_max = a.hl_max;
    g.R_max = a.R_max;
    g.sf64 = 1.0;
    g.sep64 = 0.0;
    g.sf32 = 1.0f;
    g.sep32 = 0.0f;
    g.cap = 0xFFFFFFFFu;
    g.state = nullptr;
    g.inv = false;
    g.idle = false;
  }
  // role pointers of the usual orientation: probes from pr*, staged
  // neighbours from nb*
  g.hP = a.prP;
  g.hD = a.prD;
  g.hX = a.prX;
  g.hStart = a.prStart;
  g.hCount = a.prCount;
  g.nP = a.nbP;
  g.nD = a.nbD;
  g.nX = a.nbX;
  g.nStart = a.nbStart;
  g.nCount = a.nbCount;
  g.nHl = a.nbHl;
  // Lane l watches queue order l: the eight queues of this wave's XCD first
  // (starting at its own sub-queue), then those of the other XCDs.  One
  // vector load of the 64 counters finds the first queue with work left.
  const int sub0 = (blockIdx.x >> 3) & 7;
  const int my_q = (((xcd + (threadIdx.x >> 3)) & 7) << 3) | ((sub0 + (int)threadIdx.x) & 7);
  // queue q: the items of cells [W q / 64, W (q + 1) / 64), from k_items's
  // list, or (no list) the cells themselves, one item each
  const uint32_t my_c0 = (uint32_t)(((uint64_t)W * (uint32_t)my_q) / QUEUES_PER_KERNEL);
  const uint32_t my_c1 = (uint32_t)(((uint64_t)W * (uint32_t)(my_q + 1)) / QUEUES_PER_KERNEL);
  const uint32_t my_qb = a.items ? my_c0 * a.npmax : my_c0;
  const uint32_t my_qn = a.items ? a.qcnt[my_q] : my_c1 - my_c0;
  // the first pre items of each queue belong to its own waves, one each: a
  // short launch needs no queue grab to begin
  const uint32_t pre = gridDim.x / QUEUES_PER_KERNEL;
  const uint32_t rank = blockIdx.x / QUEUES_PER_KERNEL;
  bool first = rank < pre;
  for (;;) {
    int pick = 0;  // uniform
    if (!first) {
      const uint32_t seen =
          __hip_atomic_load(&a.qctr[my_q * QSTRIDE], __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT);
      const unsigned long long open = __ballot(seen + pre < my_qn);
      if (open == 0ull) break;
      pick = (int)__builtin_ctzll(open);
    }
    const int q = __builtin_amdgcn_readlane(my_q, pick);
    const uint32_t qb = uni((uint32_t)__builtin_amdgcn_readlane((int)my_qb, pick));
    const uint32_t qn = uni((uint32_t)__builtin_amdgcn_readlane((int)my_qn, pick));
    for (;;) {
      uint32_t item = rank;
      if (!first) {
        // lane 0 takes the next item; readfirstlane makes it a scalar, so the
        // loop exit below is uniform
        uint32_t old = 0u;
        if (l0) old = atomicAdd(&a.qctr[q * QSTRIDE], 1u);
        item = uni(old) + pre;
      }
      first = false;
      if (item >= qn) break;
      uint32_t gc = qb + item, cg = 0u, ncg = 1u, sp = 0u, nst = 1u;
      if (a.items) {
        const uint2 w = a.items[qb + item];
        gc = uni(w.x);
        const uint32_t code = uni(w.y);
        cg = code & 0xFFu;
        ncg = (code >> 8) & 0xFFu;
        sp = (code >> 16) & 0xFFu;
        nst = code >> 24;
      }
      if (GEN) {
        const uint32_t inst = uni(a.cell_inst[gc]);
        if (inst != cur_inst) {
          if (cur_inst != 0xFFFFFFFFu) flush<GEN>(a, g, acc, MODE);
          const InstDesc& d = a.desc[inst];
          for (int dd = 0; dd < 3; ++dd) {
            g.box[dd] = d.smp.box[dd];
            g.boxf[dd] = d.boxf[dd];
            g.nc[dd] = d.ncell[dd];
            g.rnc[dd] = 1.0f / (float)d.ncell[dd];
            g.edge[dd] = d.edge[dd];
          }
          g.cell_base = d.cell_base;
          g.st = a.stencil + (MODE == PM_GEN_NEW ? d.hst_off : d.st_off);
          g.st_n = MODE == PM_GEN_NEW ? d.hst_n : d.st_n;
          g.ew = d.ew;
          g.hl_max = d.hl_max;
          g.R_max = d.R_max;
          g.sf64 = d.sf64;
          g.sep64 = d.sep64;
          g.sf32 = d.sf32;
          g.sep32 = d.sep32;
          g.cap = d.cap;
          g.state = &a.st[inst];
          cur_inst = inst;
          if (MODE == PM_GEN_OLD) {
            const OldRoles r = old_roles(a, inst, d);
            g.inv = uni(r.inv ? 1u : 0u) != 0u;
            g.idle = uni(r.idle ? 1u : 0u) != 0u;
            g.hP = g.inv ? a.nbP : a.prP;
            g.hD = g.inv ? a.nbD : a.prD;
            g.hX = g.inv ? a.nbX : a.prX;
            g.hStart = g.inv ? a.nbStart : a.prStart;
            g.hCount = g.inv ? a.nbCount : a.prCount;
            g.nP = g.inv ? a.prP : a.nbP;
            g.nD = g.inv ? a.prD : a.nbD;
            g.nX = g.inv ? a.prX : a.nbX;
            g.nStart = g.inv ? a.prStart : a.nbStart;
            g.nCount = g.inv ? a.prCount : a.nbCount;
            g.nHl = g.inv ? a.prHl : a.nbHl;
          } else {
            g.inv = false;
            g.idle = false;
          }
        }
      }
      process_cell<MODE, PREC, ALL>(a, g, gc, cg, ncg, sp, nst, L, acc);
    }
  }
  if (!GEN || cur_inst != 0xFFFFFFFFu) flush<GEN>(a, g, acc, MODE);
}

// Work list of a generation pass: per queue range of cells, the items of its
// cells that hold probes (and whose instance has pairs), costliest first, so
// that each queue starts with its costliest items and the launch ends on
// light ones.
//
// A cell's cost is its probes times the rods its walk is expected to stage:
// the volume of the walk (a cube of edge two reaches plus a cell edge, less
// its corners) times the mean of the cell's own neighbour density and the
// instance's.  A cell is dealt over ceil(cost / share) items: share is the
// launch's whole cost over ITEMS_PER_WAVE items per wave of the grid, but at
// least ITEM_FULL pairs, so that an item's own overhead (queue grab, probe
// loads, stencil look-up) stays small, or, where that would leave waves
// without an item, one wave's part of the cost down to ITEM_MIN pairs.
// Chunks of probes are dealt first: they share no staging anyway.  Two cost
// buckets per octave; the order inside a bucket is arbitrary, as every result
// of a pair pass is independent of the order of its work.
//
// What bounds a launch over few cells is the longest cell on one wave: 125
// cells of 160 rods kept 125 to 250 of the 4096 waves busy.  Measured on
// MI355X against one item per cell (at most two for the reject-vs-accepted
// pass), whole generations: 20,000 rods on 1 um cells, FP64, 10.2 -> 3.9 ms;
// 2,000 rods 1.84 -> 0.72 ms; 32 uneven packings 244 -> 153 ms, where empty
// cells had also been taken one by one; 500,000 and 4M rods unchanged.
// 2, 8 and 16 items per wave: the 32 packings 156, 164 and 191 ms.
constexpr int ITEM_BUCKETS = 48;
constexpr int ITEM_THREADS = 512;
constexpr float ITEMS_PER_WAVE = 4.0f;
constexpr float ITEM_MIN = 4096.0f, ITEM_FULL = 16384.0f;

struct ItemPlan {
  uint32_t ncg, nst, bucket;
};

// Walk volume of a cell whose longest probe has half length h, over the box.
__device__ __forceinline__ float walk_share(const InstDesc& d, float h) {
  float v = 0.8f;
#pragma unroll
  for (int k = 0; k < 3; ++k) {
    const float e = 2.0f * (h + d.hl_max + d.R_max) + d.edge[k];
    v *= e / d.boxf[k];
  }
  return v;
}

template <int MODE>
__device__ __forceinline__ bool item_plan(const PairArgs& a, uint32_t c, float share, ItemPlan* o) {
  const uint32_t inst = a.cell_inst[c];
  const InstDesc& d = a.desc[inst];
  uint32_t pc, nb, total;
  float h;
  if (MODE == PM_GEN_OLD) {
    const OldRoles r = old_roles(a, inst, d);
    if (r.idle) return false;
    pc = min(r.inv ? a.nbCount[c] : a.prCount[c], r.inv ? d.cap : 0xFFFFFFFFu);
    nb = r.inv ? a.prCount[c] : a.nbCount[c];
    total = r.inv ? r.nprop : r.nacc;
    h = r.inv ? a.nbHl[c] : a.prHl[c];
  } else {
    if (a.skip_walk && d.fine.on) return false;
    pc = nb = a.prCount[c];
    total = a.prStart[d.cell_base + d.ncells] - a.prStart[d.cell_base];
    h = a.prHl[c];
  }
  if (pc == 0u) return false;
  float w = (float)pc * walk_share(d, h) * 0.5f * ((float)total + (float)nb * (float)d.ncells);
  if (MODE == PM_GEN_NEW) w *= 0.5f;  // half stencil
  const uint32_t np = (uint32_t)fminf(ceilf(w / share), (float)a.npmax);
  const uint32_t nch = (pc + WAVE - 1u) / WAVE;
  o->ncg = max(1u, min(nch, np));
  const uint32_t st_n = MODE == PM_GEN_NEW ? d.hst_n : d.st_n;
  o->nst = max(1u, min(np / o->ncg, min(st_n, 255u)));
  if (a.split_min != 0u) {
    // the handle's own split (NF_OPT_PART_SHIFT, NF_OPT_SPLIT_MIN): at most
    // npmax stencil parts of at least split_min probes each
    o->ncg = 1u;
    o->nst = max(1u, min(a.npmax, (pc + a.split_min - 1u) / a.split_min));
  }
  w /= (float)(o->ncg * o->nst);
  // (bits >> 22) = 2 * biased exponent + first mantissa bit; bucket 0: w >= 2^24
  const int k = 2 * (127 + 24) - (int)(__float_as_uint(w) >> 22);
  o->bucket = (uint32_t)min(max(k, 0), ITEM_BUCKETS - 1);
  return true;
}

template <int MODE>
__global__ void __launch_bounds__(ITEM_THREADS) k_items(PairArgs a, float waves) {
  __shared__ uint32_t slot[ITEM_BUCKETS];
  __shared__ float part[ITEM_THREADS / WAVE];
  const uint32_t r = blockIdx.x;
  const uint32_t c0 = (uint32_t)(((uint64_t)a.ncells_total * r) / QUEUES_PER_KERNEL);
  const uint32_t c1 = (uint32_t)(((uint64_t)a.ncells_total * (r + 1u)) / QUEUES_PER_KERNEL);
  if (threadIdx.x < ITEM_BUCKETS) slot[threadIdx.x] = 0u;
  // the launch's whole cost, from the instances' totals
  float sum = 0.0f;
  for (int i = threadIdx.x; i < a.n_inst; i += ITEM_THREADS) {
    const InstDesc& d = a.desc[i];
    if (MODE == PM_GEN_OLD) {
      const OldRoles o = old_roles(a, (uint32_t)i, d);
      if (!o.idle) sum += (float)o.nacc * (float)o.nprop * walk_share(d, d.hl_max);
    } else {
      if (a.skip_walk && d.fine.on) continue;
      const float n = (float)(a.prStart[d.cell_base + d.ncells] - a.prStart[d.cell_base]);
      sum += 0.5f * n * n * walk_share(d, d.hl_max);
    }
  }
#pragma unroll
  for (int o = 32; o > 0; o >>= 1) sum += __shfl_xor(sum, o, WAVE);
  if ((threadIdx.x & (WAVE - 1)) == 0) part[threadIdx.x / WAVE] = sum;
  __syncthreads();
  sum = 0.0f;
  for (int k = 0; k < ITEM_THREADS / WAVE; ++k) sum += part[k];
  const float share = fmaxf(sum / (waves * ITEMS_PER_WAVE), fminf(fmaxf(sum / waves, ITEM_MIN), ITEM_FULL));
  ItemPlan p;
  for (uint32_t c = c0 + threadIdx.x; c < c1; c += ITEM_THREADS)
    if (item_plan<MODE>(a, c, share, &p)) atomicAdd(&slot[p.bucket], p.ncg * p.nst);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t at = 0;
    for (int k = 0; k < ITEM_BUCKETS; ++k) {
      const uint32_t t = slot[k];
      slot[k] = at;
      at += t;
    }
    a.qcnt[r] = at;
  }
  __syncthreads();
  uint2* out = a.items + (uint64_t)c0 * a.npmax;
  for (uint32_t c = c0 + threadIdx.x; c < c1; c += ITEM_THREADS) {
    if (!item_plan<MODE>(a, c, share, &p)) continue;
    uint32_t at = atomicAdd(&slot[p.bucket], p.ncg * p.nst);
    for (uint32_t sp = 0; sp < p.nst; ++sp)
      for (uint32_t cg = 0; cg < p.ncg; ++cg)
        out[at++] = make_uint2(c, cg | (p.ncg << 8) | (sp << 16) | (p.nst << 24));
  }
}

// Items per cell at most: about 2^19 list entries in all, between 2 and 64
// per cell.
uint32_t pair_items_max(uint64_t ncells) {
  const uint64_t k = ((uint64_t)1 << 19) / (ncells ? ncells : 1);
  return (uint32_t)(k < 2 ? 2 : (k > 64 ? 64 : k));
}

static int g_cus = 0;

int pair_grid(int mode) {
  if (g_cus == 0) {
    int dev = 0, cus = 0;
    if (hipGetDevice(&dev) != hipSuccess ||
        hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) != hipSuccess ||
        cus <= 0)
      cus = 256;
    g_cus = cus;
  }
  (void)mode;
  return g_cus * 16;
}

void launch_pair(int mode, int prec, const PairArgs& args, hipStream_t s, const PairTiles* t) {
  // the handle's tuned launch shape where set (nanofiller_amd/autotune.py)
  uint32_t waves = 0;
  if (t) waves = mode == PM_GEN_OLD ? t->waves_old : (mode == PM_GEN_NEW ? t->waves_new : 0u);
  const int cus = pair_grid(mode) / 16;
  const dim3 grid(waves ? (uint32_t)cus * waves : (uint32_t)pair_grid(mode)), block(PAIR_THREADS);
  PairArgs a = args;
  if (a.items != nullptr) {
    a.npmax = pair_items_max(a.ncells_total);
    a.split_min = 0u;
    if (t && mode == PM_GEN_OLD && (t->part_shift >= 0 || t->split_min != 0u)) {
      a.split_min = t->split_min ? t->split_min : 32u;
      a.npmax = min(a.npmax, 1u << (t->part_shift >= 0 ? t->part_shift : 1));
    }
    if (mode == PM_GEN_OLD)
      hipLaunchKernelGGL(k_items<PM_GEN_OLD>, dim3(QUEUES_PER_KERNEL), dim3(ITEM_THREADS), 0, s, a, (float)grid.x);
    else
      hipLaunchKernelGGL(k_items<PM_GEN_NEW>, dim3(QUEUES_PER_KERNEL), dim3(ITEM_THREADS), 0, s, a, (float)grid.x);
  }
  const bool all = t && t->test_all;
#define NF_LAUNCH(M, P, A) hipLaunchKernelGGL((k_pair<M, P, A>), grid, block, 0, s, a)
#define NF_LAUNCH_ALL(M, P) \
  if (all)                  \
    NF_LAUNCH(M, P, true);  \
  else                      \
    NF_LAUNCH(M, P, false)
  if (prec == NF_PREC_FP64) {
    switch (mode) {
      case PM_GEN_OLD: NF_LAUNCH_ALL(PM_GEN_OLD, NF_PREC_FP64); break;
      case PM_GEN_NEW: NF_LAUNCH_ALL(PM_GEN_NEW, NF_PREC_FP64); break;
      default: NF_LAUNCH(PM_CNT, NF_PREC_FP64, true); break;
    }
  } else {
    switch (mode) {
      case PM_GEN_OLD: NF_LAUNCH_ALL(PM_GEN_OLD, NF_PREC_FP32_RECHECK); break;
      case PM_GEN_NEW: NF_LAUNCH_ALL(PM_GEN_NEW, NF_PREC_FP32_RECHECK); break;
      default: NF_LAUNCH(PM_CNT, NF_PREC_FP32_RECHECK, true); break;
    }
  }
#undef NF_LAUNCH_ALL
#undef NF_LAUNCH
}

}  // namespace nf
