// nf_walk.hip - the generation's two rejection passes over crossing lists.
//
// An instance with crossing lists has a fine grid of about one rod per cell.
// Every accepted rod (and, per round, every survivor of the first pass) is
// entered in the list of each fine cell that its capsule of half the cut
// distance can touch.  Two rods that overlap do so around the midpoint of
// their closest points, which lies within half the cut distance of both
// axes: both are in the list of the cell that holds it.  A proposal therefore
// meets every rod it overlaps by reading the lists of the cells it crosses
// itself, a few rods each, where the cell-pair engine (nf_pair.hip) stages
// every rod whose centre may lie within reach.
//
// The passes replace the reference's kernels as nf_pair.hip does; every
// decision is the same (the rules, the FP32 band and the canonical FP64
// evaluation are those of nf_pair.hip), so a packing does not depend on which
// engine tests its pairs.
//
// nf_contacts reads contacts from the same lists, all rods entered with half
// the contact distance: a pair is taken up by the rod further on in the cell
// list and reported in the one cell that holds the midpoint of its closest
// points (nf_seg.h's rule).
//
// What bounds them: the walk is VALU issue and the latency of its fetches (at
// most 144 of a launch's 250 us issue on 32 jamming packings; 96% of its lines
// come from L2), entering is the rate of device-scope atomics, about 30 G/s.
// Whole generations on MI355X, cell-pair engine with the line filter against
// this: 500,000 log-normal rods in agglomerates 3.24 -> 1.95 ms, 20,000 rods in
// FP64 on 1 um cells 3.6 -> 1.4 ms, 32 uneven packings, some past jamming, 155 ->
// 63 ms.  Which packings take the lists: plan_fine (nf_api.cpp).
#include "nf_internal.h"
#include "nf_line.h"

namespace nf {

namespace {

// List entry: the rod's index from the instance's first (26 bits) and the
// image in which it crosses the cell (2 bits per axis, image + 1).  The rods
// themselves are read through it from one array in centre-cell order, centre
// and direction side by side, which a wave's neighbours share in L2: whole
// rods in the lists (32 bytes, each rod some twenty times) made the walk of
// 32 packings wait for random lines of a gigabyte, 0.41 ms per round.
constexpr uint32_t ENT_BITS = ENTRY_BITS;
constexpr uint32_t ENT_MASK = (1u << ENT_BITS) - 1u;

__device__ __forceinline__ uint32_t wuni(uint32_t v) { return (uint32_t)__builtin_amdgcn_readfirstlane((int)v); }

__device__ __forceinline__ uint32_t wprefix(unsigned long long mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

__device__ __forceinline__ int at3(int a, int x, int y, int z) { return a == 0 ? x : (a == 1 ? y : z); }
__device__ __forceinline__ float at3(int a, float x, float y, float z) { return a == 0 ? x : (a == 1 ? y : z); }

// Calls f(cell, image) with the fine cells that the rod's capsule of radius
// g.r may touch, in a fixed order: per slab of the rod's dominant axis the
// part of the axis within r of the slab, and the rectangle of cells its other
// two coordinates span, widened by r.  cell: index in the instance's grid;
// image: 2 bits per axis, the box edges from the cell to where the rod
// crosses it, plus 1.
template <class F>
__device__ __forceinline__ void crossed_cells(const FineGrid& g, const float4 P, const float4 D, F f) {
  const float ax = fabsf(D.x), ay = fabsf(D.y), az = fabsf(D.z);
  const int a = ax >= ay && ax >= az ? 0 : (ay >= az ? 1 : 2);
  const int b = a == 0 ? 1 : 0, c = a == 2 ? 1 : 2;
  const float pa = at3(a, P.x, P.y, P.z), pb = at3(b, P.x, P.y, P.z), pc = at3(c, P.x, P.y, P.z);
  const float ua = at3(a, D.x, D.y, D.z), ub = at3(b, D.x, D.y, D.z), uc = at3(c, D.x, D.y, D.z);
  const float ea = at3(a, g.e[0], g.e[1], g.e[2]);
  const float ia = at3(a, g.ie[0], g.ie[1], g.ie[2]);
  const float ib = at3(b, g.ie[0], g.ie[1], g.ie[2]);
  const float ic = at3(c, g.ie[0], g.ie[1], g.ie[2]);
  const int na = at3(a, g.n[0], g.n[1], g.n[2]), nb = at3(b, g.n[0], g.n[1], g.n[2]),
            nc = at3(c, g.n[0], g.n[1], g.n[2]);
  const uint32_t ta = at3(a, 1, g.n[0], g.n[0] * g.n[1]), tb = at3(b, 1, g.n[0], g.n[0] * g.n[1]),
                 tc = at3(c, 1, g.n[0], g.n[0] * g.n[1]);
  const float ha = P.w * fabsf(ua) + g.r;
  const float iu = recip(ua);
  const int k1 = (int)floorf((pa + ha) * ia);
  for (int k = (int)floorf((pa - ha) * ia); k <= k1; ++k) {
    float s0 = (((float)k * ea - g.r) - pa) * iu, s1 = (((float)(k + 1) * ea + g.r) - pa) * iu;
    const float lo = fmaxf(fminf(s0, s1), -P.w), hi = fminf(fmaxf(s0, s1), P.w);
    const float b0 = fmaf(lo, ub, pb), b1 = fmaf(hi, ub, pb);
    const float c0 = fmaf(lo, uc, pc), c1 = fmaf(hi, uc, pc);
    const int i1 = (int)floorf((fmaxf(b0, b1) + g.r) * ib);
    const int j0 = (int)floorf((fminf(c0, c1) - g.r) * ic), j1 = (int)floorf((fmaxf(c0, c1) + g.r) * ic);
    // a rod reaches less than one box edge past the box (FineGrid)
    const int wk = k < 0 ? 0 : (k >= na ? 2 : 1);
    const uint32_t ck = (uint32_t)(k - (wk - 1) * na) * ta;
    for (int i = (int)floorf((fminf(b0, b1) - g.r) * ib); i <= i1; ++i) {
      const int wi = i < 0 ? 0 : (i >= nb ? 2 : 1);
      const uint32_t ci = ck + (uint32_t)(i - (wi - 1) * nb) * tb;
      for (int j = j0; j <= j1; ++j) {
        const int wj = j < 0 ? 0 : (j >= nc ? 2 : 1);
        f(ci + (uint32_t)(j - (wj - 1) * nc) * tc,
          (uint32_t)wk << (2 * a) | (uint32_t)wi << (2 * b) | (uint32_t)wj << (2 * c));
      }
    }
  }
}

// ---------------------------------------------------------------------------
// Entering rods in the lists.  LANES lanes per rod: each walks the rod's
// cells and enters it in every LANES-th one, so that the atomics of a rod,
// which answer from beyond the XCD's L2, are in flight together.
// ---------------------------------------------------------------------------
constexpr int ENTER_LANES = 8;
constexpr int ENTER_THREADS = 256;

__device__ __forceinline__ void enter(const FineGrid& g, uint32_t* __restrict__ count, uint32_t* __restrict__ list,
                                      uint64_t off, uint32_t cap, const float4 P, const float4 D, uint32_t idx,
                                      uint32_t* overflow, uint32_t bit) {
  const uint32_t sub = threadIdx.x & (ENTER_LANES - 1);
  uint32_t ord = 0;
  bool over = false;
  crossed_cells(g, P, D, [&](uint32_t cell, uint32_t image) {
    if ((ord++ & (ENTER_LANES - 1)) != sub || over) return;
    const uint32_t gc = g.base + cell;
    const uint32_t at = atomicAdd(&count[gc], 1u);
    if (at < cap) {
      list[off + (uint64_t)cell * cap + at] = idx | image << ENT_BITS;
    } else {
      // no room: the instance stops and the host generates it again with
      // longer lists (a contact pass takes another way); readers take at most
      // cap entries of a list, and what is not entered any more does not count
      over = true;
      if ((__hip_atomic_load(overflow, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_AGENT) & bit) == 0u) atomicOr(overflow, bit);
    }
  });
}

// Survivors of the first pass, for the same-round pass.
__global__ void __launch_bounds__(ENTER_THREADS) k_enter_survivors(WalkArgs a) {
  const uint32_t total = a.prStart[a.ncells];
  for (uint64_t t = (uint64_t)blockIdx.x * ENTER_THREADS + threadIdx.x; t < (uint64_t)total * ENTER_LANES;
       t += (uint64_t)gridDim.x * ENTER_THREADS) {
    const uint32_t k = (uint32_t)(t / ENTER_LANES);
    const uint32_t inst = a.n_inst == 1 ? 0u : a.cell_inst[a.scell[a.prX[k]]];
    const InstDesc& d = a.desc[inst];
    if (!d.fine.on) continue;
    enter(d.fine, a.fcountP, a.flistP, d.fine.offP, d.fine.capP, a.prP[k], a.prD[k], k - a.prStart[d.cell_base],
          &a.st[inst].overflow, OVER_LISTS_P);
  }
}

// The instance reaches its target in this round: nothing will read its lists
// of accepted rods.
__device__ __forceinline__ bool last_round(const WalkArgs& a, const InstDesc& d, uint32_t inst) {
  const uint32_t g = a.slot_base[inst];
  return a.srank[g + a.st[inst].M] - a.srank[g] >= d.n_target - a.st[inst].n_acc;
}

// Rods accepted by this round's commit, found among the survivors of the
// first pass: these are in cell order, so that neighbouring lanes' atomics
// and stores fall into the same few lists.  In the last round nothing is
// entered (last_round).
__global__ void __launch_bounds__(ENTER_THREADS) k_enter_accepted(WalkArgs a) {
  const uint32_t total = a.prStart[a.ncells];
  for (uint64_t t = (uint64_t)blockIdx.x * ENTER_THREADS + threadIdx.x; t < (uint64_t)total * ENTER_LANES;
       t += (uint64_t)gridDim.x * ENTER_THREADS) {
    const uint32_t k = (uint32_t)(t / ENTER_LANES);
    const uint32_t slot = a.prX[k];
    if (!a.surv[slot]) continue;
    const uint32_t dst = a.sdst[slot];
    if (dst == 0xFFFFFFFFu) continue;  // past the target, or its cell was full
    const uint32_t inst = a.n_inst == 1 ? 0u : a.cell_inst[a.scell[slot]];
    const InstDesc& d = a.desc[inst];
    if (!d.fine.on || last_round(a, d, inst)) continue;
    enter(d.fine, a.fcountA, a.flistA, d.fine.offA, d.fine.capA, a.prP[k], a.prD[k], (uint32_t)(dst - d.old_off),
          &a.st[inst].overflow, OVER_LISTS_A);
  }
}

// The rods of a contact pass, all of a cell list; also side by side in rods.
__global__ void __launch_bounds__(ENTER_THREADS) k_enter_contacts(WalkArgs a) {
  const WalkContacts& c = a.cnt;
  for (uint64_t t = (uint64_t)blockIdx.x * ENTER_THREADS + threadIdx.x; t < (uint64_t)c.n * ENTER_LANES;
       t += (uint64_t)gridDim.x * ENTER_THREADS) {
    const uint32_t k = (uint32_t)(t / ENTER_LANES);
    const float4 P = c.cP[k], D = c.cD[k];
    if ((threadIdx.x & (ENTER_LANES - 1)) == 0u) {
      c.rods[2ull * k] = P;
      c.rods[2ull * k + 1u] = D;
    }
    enter(c.fine, a.fcountA, a.flistA, c.fine.offA, c.fine.capA, P, D, k, c.overflow, 1u);
  }
}

// ---------------------------------------------------------------------------
// The walk.  A wave holds 64 >> sb probes, 1 << sb lanes each (more lanes per
// probe where the launch has few).  The lanes list the cells their probe
// crosses in LDS, read the lists' lengths, then go through the lists four
// entries at a time: ids, then the four rods in flight together, then the
// line filter (nf_line.h) about the probe's centre.  The pairs it leaves
// queue in LDS and run 64 at a time through the FP32 band or FP64.  A cut
// proposal leaves; the lanes that run out of entries wait until REFILL do and
// then take the next probes, so that the few proposals that overlap nothing,
// whose lists are read to the end, do not hold the others' lanes.
// ---------------------------------------------------------------------------
constexpr int WSEG = 16;         // cells listed per lane at a time
constexpr int REFILL = 16;       // lanes without entries that make a refill worth its flush
constexpr uint32_t QFLUSH = 8;   // queued pairs that are tested at the end of a step: a cut found early saves steps
constexpr int WQ = 2 * WAVE;     // fewer than 64 wait between pushes of up to 64

struct WalkLds {
  uint32_t seg[WSEG][WAVE];   // cell | image << 26
  uint16_t len[WSEG][WAVE];   // entries in its list
  float4 sP[WAVE], sD[WAVE];  // the wave's probes
  uint32_t hit[WAVE];
  uint32_t qe[WQ], qp[WQ];    // queued pairs: rod; probe | image << 8 (contacts: entry; probe)
  uint32_t qc[WQ];            // contacts: the cell they met in, with the probe's image
};

struct WalkAcc {
  uint32_t tests, rech;
  double maxdd;
};

__device__ __forceinline__ int rel_img(uint32_t probe, uint32_t entry, int k) {
  return (int)((probe >> (2 * k)) & 3u) - (int)((entry >> (2 * k)) & 3u);
}

// One queued pair (valid lanes only): the FP32 band with FP64 recheck, or
// plain FP64, in the canonical orientation (nf_pair.hip): the proposal first,
// and of two proposals the later slot, which is the probe.
template <int PREC>
__device__ __forceinline__ void walk_full(const WalkArgs& a, const InstDesc& d, const float4* __restrict__ rods,
                                          WalkLds& L, uint32_t e, bool valid, WalkAcc& acc) {
  const uint32_t at = L.qe[e], code = L.qp[e];
  const uint32_t p = code & 0xFFu;
  const float4 P1 = L.sP[p], D1 = L.sD[p];
  if (!valid) return;
  const float4 P2 = rods[2ull * at];
  float4 D2 = rods[2ull * at + 1u];
  D2.w = D1.w;  // a packing's rods share their radius
  const int ix = (int)((code >> 8) & 7u) - 2, iy = (int)((code >> 11) & 7u) - 2, iz = (int)((code >> 14) & 7u) - 2;
  const double sx = (double)ix * d.smp.box[0], sy = (double)iy * d.smp.box[1], sz = (double)iz * d.smp.box[2];
  const double R64 = d.sf64 * ((double)D1.w + (double)D2.w) + d.sep64;
  bool cut, within = true;
  if (PREC == NF_PREC_FP64) {
    const double d2 = pair_d2_f64(P1, D1, P2, D2, sx, sy, sz, R64, &within);
    cut = within && d2 < R64 * R64;
  } else {
    const float R32 = d.sf32 * (D1.w + D2.w) + d.sep32;
    const F32Pair r = pair_f32(P1, D1, P2, D2, (float)sx, (float)sy, (float)sz, R32, d.ew, true);
    if (r.decided < 0) {
      ++acc.rech;
      const double d2 = pair_d2_f64(P1, D1, P2, D2, sx, sy, sz, R64, &within);
      cut = within && d2 < R64 * R64;
    } else {
      cut = r.decided != 0;
      if (a.diag && r.within) {
        const double e64 = pair_d2_f64(P1, D1, P2, D2, sx, sy, sz, R64, &within);
        const double dd = fabs(sqrt((double)r.d2) - sqrt(e64));
        acc.maxdd = dd > acc.maxdd ? dd : acc.maxdd;
      }
    }
  }
  if (cut) L.hit[p] = 1u;
}

// One queued pair of a contact pass (valid lanes only): the screen, band and
// reporting rule of the footprint pass (nf_seg.h); appends a contact.
__device__ __forceinline__ uint32_t crossing_translate(uint32_t image) {
  return seg_pack(1 - (int)(image & 3u), 1 - (int)((image >> 2) & 3u), 1 - (int)((image >> 4) & 3u));
}

template <int PREC>
__device__ __forceinline__ void walk_contact(const WalkContacts& c, WalkLds& L, uint32_t e, bool valid,
                                             WalkAcc& acc) {
  const uint32_t ent = L.qe[e], p = L.qp[e], cell = L.qc[e];
  const float4 P1 = L.sP[p], D1 = L.sD[p];
  const uint32_t k = L.hit[p];
  if (!valid) return;
  const uint32_t idx = ent & ENT_MASK;
  const float4 P2 = c.rods[2ull * idx], D2 = c.rods[2ull * idx + 1u];
  const uint32_t m1 = crossing_translate(cell >> ENT_BITS), m2 = crossing_translate(ent >> ENT_BITS);
  const int code = seg_screen<PREC>(c.x, P1, D1, m1, P2, D2, m2, acc.tests);
  if (code == 0) return;
  SegHit hit;
  if (!seg_full<PREC>(c.x, c.g, c.cid[k], P1, D1, m1, c.cid[idx], P2, D2, m2, cell & ENT_MASK, code, acc.tests,
                      acc.rech, acc.maxdd, &hit))
    return;
  const uint32_t pos = atomicAdd(c.app_n, 1u);
  if (pos >= c.app_cap) return;
  c.outI[pos] = hit.I;
  c.outJ[pos] = hit.J;
  c.outGap[pos] = (float)hit.gap;
  c.outGap64[pos] = hit.gap;
  c.outImg[pos] = hit.img;
}

template <int MODE, int PREC>
__global__ void __launch_bounds__(WAVE, 4) k_walk(WalkArgs a) {
  __shared__ WalkLds L;
  constexpr bool CNT = MODE == PM_CNT;
  if (!CNT && wuni(a.ri->T) == 0u) return;
  if (CNT && wuni(*a.cnt.overflow) != 0u) return;  // a list was too short: another engine's pass
  if (MODE == PM_GEN_OLD && wuni(a.ri->old) == 0u) return;
  const uint32_t lane = threadIdx.x;
  const uint32_t total = CNT ? a.cnt.n : wuni(a.prStart[a.ncells]);
  // lanes per probe: more where that leaves a wave fewer than two turns
  int sb = 0;
  while (sb < 3 && ((uint64_t)total << sb) < (uint64_t)gridDim.x * (2u * WAVE)) ++sb;
  const uint32_t per = (uint32_t)WAVE >> sb;
  const uint32_t pl = lane >> sb, sub = lane & ((1u << sb) - 1u);
  const unsigned long long group = ((1ull << (1u << sb)) - 1ull) << (pl << sb);
  const uint32_t nch = (total + per - 1u) / per;
  // proposals are in cell order: each XCD takes chunks from its own eighth of
  // them first, so that the lists and rods its waves read overlap in its L2
  const uint32_t xcd = blockIdx.x & 7u, W = gridDim.x >> 3;
  uint32_t turn = 0;
  // the wave's chunk [cur, end), the part of it in the present instance up to
  // part_end
  uint32_t cur = 0, end = 0, part_end = 0, inst = 0;
  bool open = true;  // chunks left
  // the lane's probe
  bool have = false;  // holds a probe whose verdict is not written yet
  bool more = false;  // more cells than were listed
  uint32_t k = 0, slot = 0, c0 = 0, nl = 0, s = 0, pos = 0, n = 0, cell = 0;
  bool live = false;
  float4 P1 = make_float4(0.f, 0.f, 0.f, 0.f), D1 = P1;
  float3 u1 = make_float3(0.f, 0.f, 0.f);  // its direction over R
  uint32_t qn = 0;
  WalkAcc acc = {0u, 0u, 0.0};
  // of the present instance
  const InstDesc* d = nullptr;
  uint32_t cap = 0;
  const uint32_t* count = nullptr;
  const uint32_t* list = nullptr;
  const float4* rods = nullptr;
  LineFilter ln = {0.0f, 0.0f};
  float lb = 0.0f;
  if (CNT) {
    cap = a.cnt.fine.capA;
    count = a.fcountA + a.cnt.fine.base;
    list = a.flistA + a.cnt.fine.offA;
    rods = a.cnt.rods;
    ln = a.cnt.ln;
    lb = -1.0f - ln.slack;
  }
  uint32_t seen = 0;  // contacts: entries read
  bool started = false;
  uint32_t kills = 0;
  auto flush_queue = [&]() {
    if (qn == 0u) return;
    __syncthreads();
    if (CNT)
      walk_contact<PREC>(a.cnt, L, min(lane, qn - 1u), lane < qn, acc);
    else
      walk_full<PREC>(a, *d, rods, L, min(lane, qn - 1u), lane < qn, acc);
    qn = 0u;
    __syncthreads();
  };
  // the lane's probe is cut
  auto verdict = [&]() {
    if (MODE == PM_GEN_OLD) {
      a.alive_out[k] = 0u;
    } else {
      a.surv[slot] = 0u;
      ++kills;
    }
  };
  auto flush_stats = [&]() {
    const unsigned long long wt = wave_sum_u64(acc.tests), wr = wave_sum_u64(acc.rech), wk = wave_sum_u64(kills);
    double v = acc.maxdd;
#pragma unroll
    for (int o = 32; o > 0; o >>= 1) v = fmax(v, __shfl_xor(v, o, WAVE));
    if (CNT) {
      const unsigned long long wb = 36ull * wave_sum_u64(seen);
      if (lane == 0u) {
        if (wt) atomicAdd(&a.cnt.ctr[0], wt);
        if (wr) atomicAdd(&a.cnt.ctr[1], wr);
        if (v > 0.0) atomicMax(&a.cnt.ctr[2], (unsigned long long)__double_as_longlong(v));
        atomicAdd(&a.cnt.ctr[3], wb);
      }
    } else if (lane == 0u) {
      InstState& st = a.st[inst];
      if (wt) atomicAdd(&st.pair_tests, wt);
      if (wr) atomicAdd(&st.rechecks, wr);
      if (wk) atomicAdd(&st.rej_new, wk);
      if (v > 0.0) atomicMax((unsigned long long*)&st.max_dd, (unsigned long long)__double_as_longlong(v));
      if (wt) atomicAdd(MODE == PM_GEN_OLD ? &st.tile_bytes : &st.tile_bytes_new, 36ull * wt);
    }
    acc = {0u, 0u, 0.0};
    kills = 0u;
  };
  for (;;) {
    // ---- probes without entries left take their next cells, or give way to
    // the next probe, when enough lanes wait
    const unsigned long long lv = __ballot(live);
    const bool idle = (lv & group) == 0ull;  // a probe's lanes wait for one another
    if (__popcll(__ballot(idle)) >= REFILL || lv == 0ull) {
      const unsigned long long mm = __ballot(more);
      const bool again = __ballot(idle && more) != 0ull;
      const bool hand = cur < part_end, swap = lv == 0ull && cur == part_end && (open || cur < end);
      if (again || hand || swap) {
        flush_queue();  // the idle probes' verdicts
        const bool hit = !CNT && idle && have && L.hit[pl] != 0u;
        const bool cont = idle && have && (mm & group) != 0ull && !hit;
        if (idle && have && !cont) {
          if (hit && sub == 0u) verdict();
          have = more = false;
        }
        if (cont) c0 += WSEG;
        if (swap && __ballot(have) == 0ull) {
          // the chunk's next instance, or the next chunk
          for (;;) {
            if (cur == end) {
              open = false;
              while (turn < 8u) {
                const uint32_t x = (xcd + turn) & 7u;
                const uint32_t lo = (uint32_t)((uint64_t)nch * x / 8u), hi = (uint32_t)((uint64_t)nch * (x + 1u) / 8u);
                // the first W chunks of an eighth belong to its own waves
                uint32_t c = 0xFFFFFFFFu;
                if (turn == 0u && !started) {
                  c = blockIdx.x >> 3;
                  started = true;
                } else if (hi - lo > W) {
                  uint32_t old = 0u;
                  if (lane == 0u) old = atomicAdd(a.qctr + x * QSTRIDE, 1u);
                  c = wuni(old) + W;
                }
                if (c < hi - lo) {
                  cur = part_end = (lo + c) * per;
                  end = min(cur + per, total);
                  open = true;
                  break;
                }
                ++turn;
              }
              if (!open) break;
            }
            if (CNT) {
              part_end = end;
              break;
            }
            const uint32_t i0 = a.n_inst == 1 ? 0u : wuni(a.cell_inst[a.scell[a.prX[cur]]]);
            const InstDesc* di = a.desc + i0;
            part_end = min(end, wuni(a.prStart[di->cell_base + di->ncells]));
            if (wuni(di->fine.on) == 0u || (MODE == PM_GEN_OLD && wuni(a.st[i0].n_acc) == 0u)) {
              cur = part_end;  // not this pass's probes
              continue;
            }
            if (d != di || i0 != inst) {
              if (d != nullptr) flush_stats();
              inst = i0;
              d = di;
              cap = MODE == PM_GEN_OLD ? d->fine.capA : d->fine.capP;
              count = (MODE == PM_GEN_OLD ? a.fcountA : a.fcountP) + d->fine.base;
              list = MODE == PM_GEN_OLD ? a.flistA + d->fine.offA : a.flistP + d->fine.offP;
              rods = a.rods + 2ull * (MODE == PM_GEN_OLD ? d->old_off : (uint64_t)a.prStart[d->cell_base]);
              ln = line_filter(d->R_max, d->ew, 2.00002f * (d->hl_max + d->R_max + 16.0f * d->ew));
              lb = -1.0f - ln.slack;
            }
            break;
          }
        }
        // ---- hand out probes
        const bool need = idle && !have;
        const unsigned long long nm = __ballot(need && sub == 0u);
        const uint32_t rank = (uint32_t)__popcll(nm & ((1ull << (pl << sb)) - 1ull));
        const bool fresh = need && rank < part_end - cur;
        if (fresh) {
          k = cur + rank;
          P1 = CNT ? rods[2ull * k] : a.prP[k];
          D1 = CNT ? rods[2ull * k + 1u] : a.prD[k];
          slot = CNT ? k : a.prX[k];
          u1 = make_float3(ln.scale * D1.x, ln.scale * D1.y, ln.scale * D1.z);
          c0 = 0u;
          have = true;
          if (sub == 0u) {
            L.sP[pl] = P1;
            L.sD[pl] = D1;
            L.hit[pl] = CNT ? k : 0u;
          }
        }
        cur += min((uint32_t)__popcll(nm), part_end - cur);
        // ---- their cells, WSEG per lane at a time, and the lists' lengths,
        // four loads in flight; empty lists leave
        if (fresh || cont) {
          uint32_t ns = 0, ord = 0;
          crossed_cells(CNT ? a.cnt.fine : d->fine, P1, D1, [&](uint32_t c, uint32_t image) {
            const uint32_t o = ord++;
            if ((o & ((1u << sb) - 1u)) != sub) return;
            const uint32_t at = (o >> sb) - c0;  // wraps below c0
            if (at < (uint32_t)WSEG) {
              L.seg[at][lane] = c | image << ENT_BITS;
              ns = at + 1u;
            }
          });
          more = ((ord + (1u << sb) - 1u - sub) >> sb) > c0 + WSEG;
          nl = 0;
          for (uint32_t t = 0; t < ns; t += 4u) {
            uint32_t c[4], m[4];
#pragma unroll
            for (int u = 0; u < 4; ++u) {
              c[u] = L.seg[min(t + (uint32_t)u, ns - 1u)][lane];
              m[u] = count[c[u] & ENT_MASK];
            }
#pragma unroll
            for (int u = 0; u < 4; ++u)
              if (t + (uint32_t)u < ns && m[u] != 0u) {
                L.seg[nl][lane] = c[u];
                L.len[nl][lane] = (uint16_t)min(m[u], cap);
                ++nl;
              }
          }
          s = pos = n = 0u;
          live = nl != 0u;
        }
        __syncthreads();
        continue;
      }
      if (lv == 0ull) break;
    }
    // ---- up to four entries of each lane's list
    if (live && pos >= n) {
      live = s < nl;
      if (live) {
        cell = L.seg[s][lane];
        n = L.len[s][lane];
        pos = 0;
        ++s;
      }
    }
    uint32_t ent[4] = {0u, 0u, 0u, 0u};
    bool may[4] = {false, false, false, false};
    if (live) {
      const uint32_t m = n - pos;  // entries left in the list
      const uint4 v = *reinterpret_cast<const uint4*>(list + (uint64_t)(cell & ENT_MASK) * cap + pos);
      ent[0] = v.x;
      ent[1] = m > 1u ? v.y : v.x;
      ent[2] = m > 2u ? v.z : v.x;
      ent[3] = m > 3u ? v.w : v.x;
      float4 P2[4], D2[4];
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        // contacts: each pair from the rod further on in the cell list, so the
        // others need not be fetched (the probe's own line is at hand)
        const uint32_t r = ent[u] & ENT_MASK;
        const float4* e = rods + 2u * (CNT ? min(r, k) : r);
        P2[u] = e[0];
        D2[u] = e[1];
      }
      // images only where an entry's differs from the cell's (rods across a face)
      const uint32_t pi = cell >> ENT_BITS;
      const uint32_t diff = ((ent[0] >> ENT_BITS) ^ pi) | ((ent[1] >> ENT_BITS) ^ pi) | ((ent[2] >> ENT_BITS) ^ pi) |
                            ((ent[3] >> ENT_BITS) ^ pi);
      if (diff != 0u) {
#pragma unroll
        for (int u = 0; u < 4; ++u) {
          const uint32_t im = ent[u] >> ENT_BITS;
          const float* bf = CNT ? a.cnt.x.boxf : d->boxf;
          P2[u].x += (float)rel_img(pi, im, 0) * bf[0];
          P2[u].y += (float)rel_img(pi, im, 1) * bf[1];
          P2[u].z += (float)rel_img(pi, im, 2) * bf[2];
        }
      }
#pragma unroll
      for (int u = 0; u < 4; ++u) {
        may[u] = (uint32_t)u < m &&
                 line_apart_from(u1, P2[u].x - P1.x, P2[u].y - P1.y, P2[u].z - P1.z, D1, D2[u], lb) < 0.0f;
        // same-round pass: only an earlier slot rejects the probe
        if (MODE == PM_GEN_NEW) may[u] = may[u] && __float_as_uint(D2[u].w) < slot;
        if (CNT) may[u] = may[u] && (ent[u] & ENT_MASK) < k;
      }
      if (CNT)
        seen += min(m, 4u);
      else
        acc.tests += min(m, 4u);
      pos += 4u;
    }
    bool ran = false;
#pragma unroll
    for (int u = 0; u < 4; ++u) {
      const unsigned long long m = __ballot(may[u]);
      if (m == 0ull) continue;
      if (may[u]) {
        const uint32_t at = qn + wprefix(m);
        const uint32_t im = ent[u] >> ENT_BITS, pi = cell >> ENT_BITS;
        if (CNT) {
          L.qe[at] = ent[u];
          L.qp[at] = pl;
          L.qc[at] = cell;
        } else {
          L.qe[at] = ent[u] & ENT_MASK;
          L.qp[at] = pl | (uint32_t)(rel_img(pi, im, 0) + 2) << 8 | (uint32_t)(rel_img(pi, im, 1) + 2) << 11 |
                     (uint32_t)(rel_img(pi, im, 2) + 2) << 14;
        }
      }
      qn += (uint32_t)__popcll(m);
      if (qn >= (uint32_t)WAVE) {
        __syncthreads();
        if (CNT)
          walk_contact<PREC>(a.cnt, L, qn - WAVE + lane, true, acc);
        else
          walk_full<PREC>(a, *d, rods, L, qn - WAVE + lane, true, acc);
        qn -= WAVE;
        __syncthreads();
        ran = true;
      }
    }
    if (!CNT && qn >= QFLUSH) {
      flush_queue();
      ran = true;
    }
    // a proposal once cut is rejected whatever else it overlaps
    if (!CNT && ran) live = live && L.hit[pl] == 0u;
  }
  if (!CNT && d == nullptr) return;
  flush_queue();
  if (!CNT && have && sub == 0u && L.hit[pl] != 0u) verdict();
  flush_stats();
}

int enter_grid(uint64_t rods) {
  uint64_t b = (rods * ENTER_LANES + ENTER_THREADS - 1) / ENTER_THREADS;
  return (int)(b > 16384 ? 16384 : (b < 1 ? 1 : b));
}

}  // namespace

void launch_enter(bool accepted, const WalkArgs& a, uint64_t rods, hipStream_t s) {
  if (accepted)
    hipLaunchKernelGGL(k_enter_accepted, dim3(enter_grid(rods)), dim3(ENTER_THREADS), 0, s, a);
  else
    hipLaunchKernelGGL(k_enter_survivors, dim3(enter_grid(rods)), dim3(ENTER_THREADS), 0, s, a);
}

void launch_enter_contacts(const WalkArgs& a, hipStream_t s) {
  hipLaunchKernelGGL(k_enter_contacts, dim3(enter_grid(a.cnt.n)), dim3(ENTER_THREADS), 0, s, a);
}

// (whole blocks per XCD: the walk deals its chunks to eighths of the grid)
void launch_walk(int mode, int prec, const WalkArgs& a, hipStream_t s, const PairTiles* t) {
  uint32_t waves = t ? (mode == PM_GEN_OLD ? t->waves_old : t->waves_new) : 0u;
  if (waves == 0u || waves > 16u) waves = 16u;
  const uint32_t blocks = (uint32_t)(pair_grid(mode) / 16) * waves;
  const dim3 grid((blocks + 7u) / 8u * 8u), block(WAVE);
  if (mode == PM_CNT) {
    if (prec == NF_PREC_FP64)
      hipLaunchKernelGGL((k_walk<PM_CNT, NF_PREC_FP64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((k_walk<PM_CNT, NF_PREC_FP32_RECHECK>), grid, block, 0, s, a);
  } else if (mode == PM_GEN_OLD) {
    if (prec == NF_PREC_FP64)
      hipLaunchKernelGGL((k_walk<PM_GEN_OLD, NF_PREC_FP64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((k_walk<PM_GEN_OLD, NF_PREC_FP32_RECHECK>), grid, block, 0, s, a);
  } else {
    if (prec == NF_PREC_FP64)
      hipLaunchKernelGGL((k_walk<PM_GEN_NEW, NF_PREC_FP64>), grid, block, 0, s, a);
    else
      hipLaunchKernelGGL((k_walk<PM_GEN_NEW, NF_PREC_FP32_RECHECK>), grid, block, 0, s, a);
  }
}

}  // namespace nf
