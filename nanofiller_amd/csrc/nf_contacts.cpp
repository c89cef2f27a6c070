// nf_contacts.cpp - host orchestration of contact detection and histograms
// on the packing of instance 0.
//
// Contacts: bin -> one pair pass (crossing lists, footprints on home cells, or
// cell pairs) that appends every contact to an unsorted list -> CSR over I (count, scan, scatter) -> canonical row sort -> contact
// areas.  This replaces the COUNT and RECORD passes of get_contact_counts /
// get_contact_arrays (src/get_contact_arrays.cu:12-140); a pass whose list
// overflows the append buffer is repeated once at the exact size.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <cstring>
#include <string>
#include <vector>

#include "nf_host.h"

using namespace nf;

namespace nf {

// Reach bounds of the contact rods: the instance's bounds after generation,
// else the largest half length and radius of the rods (one device reduction).
// dev: how far the squares of the directions are from 1 (0 for generated
// rods, whose directions are rounded unit vectors).
int contact_bounds(nf_handle* h, uint32_t n, const float4* P, const float4* D, float* hlmax, float* amax,
                   float* dev) {
  *hlmax = h->desc[h->post_inst].hl_max;
  *amax = (float)h->params[h->post_inst].radius;
  if (dev) *dev = 0.0f;
  if (h->generated) return NF_OK;
  uint32_t* out = nullptr;
  int rc = dalloc(h, &out, 4);
  if (rc != NF_OK) return rc;
  float v[3] = {0.0f, 0.0f, 0.0f};
  fill_u32(out, 0u, 4, h->stream);
  launch_rod_bounds(P, D, n, out, h->stream);
  const HostPart part = {v, out, sizeof(v)};
  hipError_t e = to_host(h, &part, 1);
  if (e == hipSuccess) e = hipGetLastError();
  dfree(h, out);
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("rod bounds: ") + hipGetErrorString(e));
  *hlmax = v[0];
  *amax = v[1];
  if (dev) *dev = v[2];
  return NF_OK;
}

static double contact_reach(const ContactBuffers& c) {
  const double Rmax = ((double)c.a_max + (double)c.a_max) + c.gap_cut;
  return ((double)c.hl_max + (double)c.hl_max) * REACH_PAD + Rmax;
}

// Scratch of bin_rods, given back by the caller once the stream has
// synchronized.
struct BinScratch {
  uint32_t* M = nullptr;
  uint32_t* tmp = nullptr;
  float4* tP = nullptr;
  float4* tD = nullptr;
  uint32_t* tid = nullptr;
};

static void free_bin_scratch(nf_handle* h, BinScratch* b) {
  dfree(h, b->M);
  dfree(h, b->tmp);
  dfree(h, b->tP);
  dfree(h, b->tD);
  dfree(h, b->tid);
  *b = BinScratch{};
}

// Cell list of n rods on the stream (launch_bin_rods): rods in cell order
// and each cell's start (ncells + 1), count and largest half length.
static int bin_rods(nf_handle* h, const float4* P, const float4* D, uint32_t n, const int32_t nc[3],
                    const double scale[3], float4* cP, float4* cD, uint32_t* cid, uint32_t* cstart,
                    uint32_t* ccount, float* chl, BinScratch* b) {
  const uint64_t ncells = (uint64_t)nc[0] * nc[1] * nc[2];
  const BinPlan bp = bin_plan(n, ncells);
  const uint64_t n1 = std::max<uint64_t>(n, 1);
  int rc = NF_OK;
  if (rc == NF_OK) rc = dalloc(h, &b->M, bp.m_words + 1);
  if (rc == NF_OK) rc = dalloc(h, &b->tmp, scan_tmp_words(bp.m_words));
  if (rc == NF_OK) rc = dalloc(h, &b->tP, n1);
  if (rc == NF_OK) rc = dalloc(h, &b->tD, n1);
  if (rc == NF_OK) rc = dalloc(h, &b->tid, n1);
  if (rc != NF_OK) return rc;
  launch_bin_rods(bp, P, D, n, nc, scale, b->M, b->tmp, b->tP, b->tD, b->tid, cP, cD, cid, cstart, ccount, chl,
                  h->stream);
  return NF_OK;
}

// Centre cell list of the contact rods on cells of about `edge`, with the
// stencil of every cell within `reach` of a home block of bx cells along x
// (half, bx = 1: each cell pair once).  The scratch is in use until the
// caller has waited for the stream and frees it.
static int build_cell_list(nf_handle* h, double edge, double reach, bool half, BinScratch* bs, int bx = 1) {
  ContactBuffers& c = h->cb;
  const nf_params& p = h->params[h->post_inst];
  const uint32_t n = c.n_rods;
  const float4* P = h->gb.bP + h->desc[h->post_inst].rod_off;
  const float4* D = h->gb.bD + h->desc[h->post_inst].rod_off;
  hipStream_t s = h->stream;
  uint64_t ncells = 1;
  double scale[3];
  for (int a = 0; a < 3; ++a) {
    double nn = std::floor(p.box[a] / edge);
    if (nn < 1.0) nn = 1.0;
    if (nn > 1024.0) nn = 1024.0;
    c.ncell[a] = (int32_t)nn;
    scale[a] = (double)c.ncell[a] / p.box[a];
    c.cscale[a] = scale[a];
    ncells *= (uint64_t)c.ncell[a];
  }
  if (ncells > (1ull << 26)) return fail(h, NF_E_INVALID, "contact grid too large");
  c.ncells = (uint32_t)ncells;
  std::vector<int4>& st = h->contact_stencil;
  st = build_stencil(c.ncell, p.box, reach, half, bx);
  c.st_n = (uint32_t)st.size();
  int rc = NF_OK;
#define ALLOC(ptr, cnt) \
  if (rc == NF_OK) rc = dalloc(h, &(ptr), (cnt));
  ALLOC(c.cP, std::max<uint64_t>(n, 1));
  ALLOC(c.cD, std::max<uint64_t>(n, 1));
  ALLOC(c.cid, std::max<uint64_t>(n, 1));
  ALLOC(c.cstart, ncells + 1);
  ALLOC(c.ccount, ncells);
  ALLOC(c.chl, ncells);
  ALLOC(c.stencil, st.size());
#undef ALLOC
  if (rc != NF_OK) return rc;
  HIPCHK(h, hipMemcpyAsync(c.stencil, st.data(), sizeof(int4) * st.size(), hipMemcpyHostToDevice, s));
  return bin_rods(h, P, D, n, c.ncell, scale, c.cP, c.cD, c.cid, c.cstart, c.ccount, c.chl, bs);
}

// Cell list of the cell-pair engine: cells of about one typical pair reach,
// half stencil of the longest pair reach.
static int contact_cells(nf_handle* h, BinScratch* bs) {
  ContactBuffers& c = h->cb;
  if (c.cP && c.cell_list == 1) return NF_OK;
  if (c.cP) {
    // the footprint engine's list (home-cell grid, run stencil): rebuild
    void* ptrs[] = {c.cP, c.cD, c.cid, c.cstart, c.ccount, c.chl, c.cmask, c.stencil};
    for (void* q : ptrs) dfree(h, q);
    c.cP = c.cD = nullptr;
    c.cid = c.cstart = c.ccount = c.cmask = nullptr;
    c.chl = nullptr;
    c.stencil = nullptr;
    c.cell_list = 0;
  }
  const nf_params& p = h->params[h->post_inst];
  const double Rmax = ((double)c.a_max + (double)c.a_max) + c.gap_cut;
  const double reach = contact_reach(c);
  // cell edge about one typical pair reach; the sorted stencil reaches the
  // longest rods and per-cell length bounds prune the rest
  double edge = (p.len_law == NF_LEN_LOGNORMAL ? p.len : (double)c.hl_max * 2.0) * REACH_PAD + Rmax;
  if (edge > reach) edge = reach;
  edge = default_cell_edge(edge, (double)c.n_rods / (p.box[0] * p.box[1] * p.box[2]), 1.0);
  const int rc = build_cell_list(h, edge, reach, true, bs);
  if (rc == NF_OK) c.cell_list = 1;
  return rc;
}

int build_contact_cells(nf_handle* h) {
  BinScratch bs;
  int rc = contact_cells(h, &bs);
  const hipError_t e = sync_stream(h->stream, "contact cell list");
  free_bin_scratch(h, &bs);
  if (rc == NF_OK && e != hipSuccess)
    rc = fail(h, NF_E_HIP, std::string("contact cell list: ") + hipGetErrorString(e));
  return rc;
}

// Footprint engine: home cells sized so that about 64 rods (the occupancy
// option) cross one at the mean density (rho (E^3 + 1.5 L E^2) rods of
// length L cross a cube of edge E, by Cauchy's mean projected area); a work
// unit that overflows its survivor table in a denser region is redone one
// cell at a time.  Fine cells of about a fifth of a rod length (the fine
// option sets the fraction) inside them.  Measured on 4M uniform 1 um rods,
// 200k 4 um rods, 500k log-normal rods in agglomerates and 8M rods in 16
// agglomerates: occupancy 32-64 and fine fraction 0.2 are within 20% of
// the best for each; from 96 on, units are redone cell by cell too often.
static void footprint_cells(nf_handle* h, uint32_t n, double* edge, int* fine) {
  const nf_params& p = h->params[h->post_inst];
  const ContactBuffers& c = h->cb;
  const double typ = p.len_law == NF_LEN_LOGNORMAL ? p.len : (double)c.hl_max * 2.0;
  const double V = p.box[0] * p.box[1] * p.box[2];
  const double rho = (double)n / V;
  const double occ = h->opt_footprint_occ > 0 ? (double)h->opt_footprint_occ : 64.0;
  double lo = 1e-3, hi = std::max(p.box[0], std::max(p.box[1], p.box[2]));
  for (int it = 0; it < 60; ++it) {
    const double e = 0.5 * (lo + hi);
    if (rho * (e * e * e + 1.5 * typ * e * e) > occ)
      hi = e;
    else
      lo = e;
  }
  *edge = std::max(lo, 4.0 * ((double)c.a_max + c.gap_cut));
  const double ff = h->opt_footprint_fine > 0 ? h->opt_footprint_fine * 1e-3 : 0.2;
  int f = (int)std::lround(*edge / std::max(typ * ff, 1e-6));
  *fine = f < 1 ? 1 : (f > 4 ? 4 : f);
}

// Ways of a contact pass.
enum ContactWay {
  WAY_LISTS,  // crossing lists (nf_walk.hip)
  WAY_SEG,    // footprints on home cells (nf_seg.hip)
  WAY_CELLS   // cell pairs (nf_pair.hip)
};

// Crossing lists of the contact rods: fine cells of 1.5 times the mean spacing
// as in generation, at least four radii wide (a_max + gap / 2).  False when
// the rods do not suit them: directions far from unit length, rods that reach
// past a box edge, radii that do not fit fine cells.
static bool contact_fine(nf_handle* h, uint32_t n, float dev, double gap, double ew, FineGrid* f, SegGrid* g) {
  const ContactBuffers& c = h->cb;
  const nf_params& p = h->params[h->post_inst];
  if (n == 0 || !(dev <= 1e-3f)) return false;
  const double V = p.box[0] * p.box[1] * p.box[2];
  const double typ = p.len_law == NF_LEN_LOGNORMAL ? rod_mean(h, h->post_inst).len : 2.0 * (double)c.hl_max;
  double E = std::min(std::max(1.5 * std::cbrt(V / (double)n), typ / 16.0), typ / 1.5);
  *g = seg_grid(p.box, E, (double)c.a_max, gap, ew);
  if (4.0 * (double)g->r > E) {
    E = 4.0 * (double)g->r;
    if (E > typ / 1.5) return false;
    *g = seg_grid(p.box, E, (double)c.a_max, gap, ew);
  }
  for (int a = 0; a < 3; ++a) {
    if (!((double)c.hl_max * 1.002 + (double)g->r < 0.999 * p.box[a])) return false;
    f->n[a] = g->nc[a];
    f->e[a] = g->h[a];
    f->ie[a] = g->inv_h[a];
  }
  if ((uint64_t)g->nc[0] * g->nc[1] * g->nc[2] > (1ull << ENTRY_BITS) || n > (1u << ENTRY_BITS)) return false;
  f->r = g->r;
  f->base = 0u;
  f->offA = 0u;
  // the plan's density peak; a list that is too short ends the pass
  const double peak = p.den_law == NF_DEN_AGGLOM ? p.agg_peak : (p.den_law == NF_DEN_MESH ? 3.0 : 1.0);
  const double lam = peak * (double)n / (double)g->ncells * 2.0 * (0.75 * typ / E + 1.0);
  f->capA = (uint32_t)std::min(4.0 * std::ceil((1.15 * lam + 6.0 * std::sqrt(lam) + 10.0) / 4.0), 8192.0);
  return (uint64_t)g->ncells * f->capA <= (1ull << 32);
}

// One contact pass.  Returns 1 (not an NF_ status) when its way does not
// suit the rods: a crossing list too short, a home cell with too many
// survivors, rods outside what the way takes.
static int contacts_pass(nf_handle* h, double gap, uint64_t* n_out, int prec, ContactWay way) {
  const bool cells = way == WAY_CELLS;
  ContactBuffers& c = h->cb;
  const nf_params& p = h->params[h->post_inst];
  const InstDesc& d = h->desc[h->post_inst];
  const uint32_t n = h->n_rods[h->post_inst];
  const float4* P = h->gb.bP + d.rod_off;
  const float4* D = h->gb.bD + d.rod_off;
  hipStream_t s = h->stream;
  // release previous results
  release_contacts(h);
  c.n_rods = n;
  c.gap_cut = gap;
  float hlmax = 0.0f, amax = 0.0f, dev = 0.0f;
  int rc = contact_bounds(h, n, P, D, &hlmax, &amax, &dev);
  if (rc != NF_OK) return rc;
  c.hl_max = hlmax;
  c.a_max = amax;
  const double Rmax = ((double)amax + (double)amax) + gap;
  const double reach = contact_reach(c);
  const double Lmax = std::max(p.box[0], std::max(p.box[1], p.box[2]));
  const double ew = 5.9604644775390625e-8 * (Lmax + reach) * 1.01;
  WalkArgs wa{};
  if (way == WAY_LISTS && !contact_fine(h, n, dev, gap, ew, &wa.cnt.fine, &wa.cnt.g)) return 1;
  float4* lrods = nullptr;
  uint32_t *lcount = nullptr, *llist = nullptr;
  bool lown = false;  // the lists are this pass's own (else the generation's, idle here)
  struct ListUse {
    nf_handle* h;
    ~ListUse() { h->lists_in_use = false; }
  } list_use{h};
  unsigned long long* ctr = nullptr;
  uint32_t* tmp = nullptr;
  uint32_t* queues = nullptr;
#define ALLOC(ptr, cnt) \
  if (rc == NF_OK) rc = dalloc(h, &(ptr), (cnt));
  ALLOC(c.cnt, (uint64_t)n + 1);
  ALLOC(c.rowptr, (uint64_t)n + 1);
  // pair tests, rechecks, max dd, tile bytes, append count, work counter, overflow; then, on lines of their
  // own (the waves that have ended add to the counters' line, 12 ns each, and a wave that takes its next item
  // must not wait behind them), the work queues
  constexpr uint64_t CTR_LINE = 2 * QSTRIDE, CTR_WORDS = CTR_LINE + 2 * QWORDS;
  ALLOC(ctr, CTR_WORDS / 2);
  ALLOC(tmp, scan_tmp_words((uint64_t)n + 1));
#undef ALLOC
  BinScratch bs;
  HostScalars* scalars = host_scalars(h);
  auto free_scratch = [&]() {
    free_bin_scratch(h, &bs);
    dfree(h, ctr);
    dfree(h, tmp);
    dfree(h, lrods);
    if (lown) {
      dfree(h, lcount);
      dfree(h, llist);
    }
    ctr = nullptr;
    tmp = queues = lcount = llist = nullptr;
    lrods = nullptr;
  };
  if (rc != NF_OK) {
    free_scratch();
    return rc;
  }
  hipEvent_t* ev = h->ev;
  hipEventRecord(ev[0], s);
  queues = (uint32_t*)ctr + CTR_LINE;
  fill_u32((uint32_t*)ctr, 0u, CTR_WORDS, s);
  PairArgs a{};
  SegCrossArgs xa{};
  // ---- bin: centre cell list
  if (cells || way == WAY_LISTS) {
    rc = contact_cells(h, &bs);
  } else {
    double edge = 0.0;
    int fine = 1;
    footprint_cells(h, n, &edge, &fine);
    c.fp_edge = edge;
    c.fp_fine = fine;
    xa.g = seg_grid(p.box, edge, (double)amax, gap, ew);
    const double rpad = (double)xa.g.r + 2.0 * (double)CELL_MARGIN;
    rc = build_cell_list(h, edge, (double)hlmax * REACH_PAD + rpad, false, &bs, SEG_ROW);
    if (rc == NF_OK) c.cell_list = 2;
    xa.fine = fine;
    xa.rpad = (float)rpad;
    const float rr = (float)((double)hlmax * REACH_PAD + rpad) * 1.0001f;
    xa.reach2 = rr * rr;
  }
  if (rc != NF_OK) {
    free_scratch();
    return rc;
  }
  if (cells) {
    a.desc = nullptr;
    a.st = nullptr;
    a.cell_inst = nullptr;
    a.ncells_total = c.ncells;
    a.stencil = c.stencil;
    a.st_off = 0;
    a.st_n = c.st_n;
    a.prP = c.cP;
    a.prD = c.cD;
    a.prX = c.cid;
    a.prStart = c.cstart;
    a.prCount = c.ccount;
    a.nbP = c.cP;
    a.nbD = c.cD;
    a.nbX = c.cid;
    a.nbStart = c.cstart;
    a.nbCount = c.ccount;
    a.nbHl = c.chl;
    a.qctr = queues;
    for (int k = 0; k < 3; ++k) {
      a.box[k] = p.box[k];
      a.boxf[k] = (float)p.box[k];
      a.ncell[k] = c.ncell[k];
    }
    a.gap64 = gap;
    a.gap32 = (float)gap;
    a.ew = (float)ew;
    a.hl_max = hlmax;
    a.R_max = (float)Rmax * 1.000001f;
    a.ctr = ctr;
    a.diag = h->opt_diag;
  } else if (way == WAY_LISTS) {
    WalkContacts& w = wa.cnt;
    const uint64_t entries = (uint64_t)w.g.ncells * w.fine.capA;
    rc = dalloc(h, &lrods, 2 * (uint64_t)n);  // (before the look at the lists: it may cost them)
    if (h->gb.walk && h->gb.total_fine >= w.g.ncells && h->gb.total_listA >= entries) {
      lcount = h->gb.fcountA;  // cleared again before the next generation
      llist = h->gb.flistA;
      h->lists_in_use = true;
    } else {
      lown = true;
      if (rc == NF_OK) rc = dalloc(h, &lcount, w.g.ncells);
      if (rc == NF_OK) rc = dalloc(h, &llist, entries);
    }
    if (rc != NF_OK) {
      free_scratch();
      return rc == NF_E_NOMEM ? 1 : rc;
    }
    for (int k = 0; k < 3; ++k) {
      w.x.box[k] = p.box[k];
      w.x.boxf[k] = (float)p.box[k];
    }
    w.x.gap64 = gap;
    w.x.gap32 = (float)gap;
    w.x.ew = (float)ew;
    w.x.diag = h->opt_diag;
    w.ln = line_filter((float)Rmax * 1.000001f, (float)ew, 2.0001f * (hlmax + (float)Rmax) + 32.0f * (float)ew, dev);
    w.n = n;
    w.cP = c.cP;
    w.cD = c.cD;
    w.cid = c.cid;
    w.rods = lrods;
    w.overflow = (uint32_t*)(ctr + 6);
    w.ctr = ctr;
    wa.fcountA = lcount;
    wa.flistA = llist;
    wa.qctr = queues;
    fill_u32(lcount, 0u, w.g.ncells, s);
    launch_enter_contacts(wa, s);
    c.fp_edge = (double)w.g.h[0];
    c.fp_fine = 1;
  } else {
    // the claim grid is the cell list's grid
    for (int k = 0; k < 3; ++k) {
      xa.g.nc[k] = c.ncell[k];
      xa.g.h[k] = (float)(p.box[k] / (double)c.ncell[k]);
      xa.g.inv_h[k] = (float)((double)c.ncell[k] / p.box[k]);
      xa.g.inv_h64[k] = (double)c.ncell[k] / p.box[k];
      xa.x.box[k] = p.box[k];
      xa.x.boxf[k] = (float)p.box[k];
    }
    xa.g.ncells = c.ncells;
    xa.cP = c.cP;
    xa.cD = c.cD;
    xa.cid = c.cid;
    xa.cstart = c.cstart;
    xa.ccount = c.ccount;
    xa.chl = c.chl;
    xa.stencil = c.stencil;
    xa.st_n = c.st_n;
    xa.x.gap64 = gap;
    xa.x.gap32 = (float)gap;
    xa.x.ew = (float)ew;
    xa.x.diag = h->opt_diag;
    xa.ctr = ctr;
    xa.next = queues;  // eight counters, QSTRIDE words apart
    xa.overflow = (uint32_t*)(ctr + 6);
    // each rod's crossing of its neighbour cells, once per rod
    rc = dalloc(h, &c.cmask, std::max<uint64_t>(n, 1));
    if (rc != NF_OK) {
      free_scratch();
      return rc;
    }
    launch_seg_marks(c.cP, c.cD, n, c.ncell, c.cscale, xa.g.h, xa.g.r, 4.0f * xa.x.ew, c.cmask, s);
    xa.cmask = c.cmask;
  }
  hipEventRecord(ev[1], s);
  // one pair pass appends every contact to an unsorted list.  Append
  // capacity: the previous call's count, else one contact per two rods; a
  // pass that overflows is repeated with the exact size
  uint64_t cap = std::max<uint64_t>(h->contact_hint + h->contact_hint / 8 + 1024, (uint64_t)n / 2 + 4096);
  if (cap > 0xFFFFFFF0ull) cap = 0xFFFFFFF0ull;
  uint32_t* appI = nullptr;
  uint32_t* appJ = nullptr;
  float* appG = nullptr;
  double* appG64 = nullptr;
  int32_t* appImg = nullptr;
  auto free_app = [&]() {
    dfree(h, appI);
    dfree(h, appJ);
    dfree(h, appG);
    dfree(h, appG64);
    dfree(h, appImg);
    appI = appJ = nullptr;
    appG = nullptr;
    appG64 = nullptr;
    appImg = nullptr;
  };
  auto free_all = [&]() {
    free_app();
    free_scratch();
  };
  uint32_t total = 0;
  for (int attempt = 0; attempt < 2; ++attempt) {
    rc = NF_OK;
    if (rc == NF_OK) rc = dalloc(h, &appI, cap);
    if (rc == NF_OK) rc = dalloc(h, &appJ, cap);
    if (rc == NF_OK) rc = dalloc(h, &appG, cap);
    if (rc == NF_OK) rc = dalloc(h, &appG64, cap);
    if (rc == NF_OK) rc = dalloc(h, &appImg, cap);
    if (rc != NF_OK) {
      free_all();
      return rc;
    }
    if (attempt > 0) {
      fill_u32((uint32_t*)ctr, 0u, CTR_WORDS, s);
    }
    hipEventRecord(ev[1], s);
    if (cells) {
      a.app_n = (uint32_t*)(ctr + 4);
      a.app_cap = (uint32_t)cap;
      a.outI = appI;
      a.outJ = appJ;
      a.outGap = appG;
      a.outGap64 = appG64;
      a.outImg = appImg;
      launch_pair(PM_CNT, prec, a, s);
    } else if (way == WAY_LISTS) {
      WalkContacts& w = wa.cnt;
      w.app_n = (uint32_t*)(ctr + 4);
      w.app_cap = (uint32_t)cap;
      w.outI = appI;
      w.outJ = appJ;
      w.outGap = appG;
      w.outGap64 = appG64;
      w.outImg = appImg;
      launch_walk(PM_CNT, prec, wa, s);
    } else {
      xa.app_n = (uint32_t*)(ctr + 4);
      xa.app_cap = (uint32_t)cap;
      xa.outI = appI;
      xa.outJ = appJ;
      xa.outGap = appG;
      xa.outGap64 = appG64;
      xa.outImg = appImg;
      launch_seg_cross(prec, xa, s);
    }
    hipEventRecord(ev[2], s);
    trace("contacts: %u rods, %s pass launched", n,
          cells ? "cell-pair" : (way == WAY_LISTS ? "crossing-list" : "footprint"));
    HIPCHK(h, scalars_to_host(h, scalars->ctr, ctr, sizeof(scalars->ctr)));
    HIPCHK(h, sync_stream(s, "contact pair pass"));
    total = (uint32_t)scalars->ctr[4];
    const uint32_t over = (uint32_t)scalars->ctr[6];
    HIPCHK(h, hipGetLastError());
    if (over) {
      trace("contacts: more rods cross a cell than fit; another engine instead");
      if (way == WAY_LISTS) h->short_gap[h->post_inst] = gap;
      free_all();
      return 1;
    }
    if ((uint64_t)total <= cap) break;
    trace("contacts: %u contacts exceed the append capacity %llu, repeating the pass", total,
          (unsigned long long)cap);
    free_app();
    cap = (uint64_t)total;
    if (attempt == 1) {
      free_all();
      return fail(h, NF_E_STATE, "contact count changed between two identical passes");
    }
  }
  h->contact_hint = total;
  c.n_contacts = total;
  c.cap_contacts = total;
  rc = NF_OK;
  if (rc == NF_OK) rc = dalloc(h, &c.I, total);
  if (rc == NF_OK) rc = dalloc(h, &c.J, total);
  if (rc == NF_OK) rc = dalloc(h, &c.gap, total);
  if (rc == NF_OK) rc = dalloc(h, &c.gap64, total);
  if (rc == NF_OK) rc = dalloc(h, &c.img, total);
  if (rc == NF_OK) rc = dalloc(h, &c.area, total);
  if (rc != NF_OK) {
    free_all();
    return rc;
  }
  // CSR over I: counts, scan, scatter, canonical row order
  hipEventRecord(ev[3], s);
  fill_u32(c.cnt, 0u, (uint64_t)n + 1, s);
  launch_csr_count(appI, total, c.cnt, s);
  scan_u32(c.cnt, c.rowptr, n, tmp, s);
  launch_csr_scatter(appI, appJ, appG, appG64, appImg, total, c.rowptr, c.cnt, c.I, c.J, c.gap, c.gap64,
                     c.img, s);
  hipEventRecord(ev[4], s);
  launch_row_sort(c.rowptr, n, c.J, c.gap, c.gap64, c.img, s);
  launch_contact_area(P, D, total, c.I, c.J, c.img, p.box, gap, c.area, s);
  hipEventRecord(ev[5], s);
  std::copy(scalars->ctr, scalars->ctr + 6, h->cb_stats);
  HIPCHK(h, sync_stream(s, "contact list"));
  trace("contacts: %u recorded and sorted", total);
  HIPCHK(h, hipGetLastError());
  float ms = 0.0f;
  const int from[4] = {0, 1, 3, 4}, to[4] = {1, 2, 4, 5};
  for (int k = 0; k < 4; ++k) {
    (void)hipEventElapsedTime(&ms, ev[from[k]], ev[to[k]]);
    h->cb_ms[k] = ms;
  }
  free_all();
  c.valid = true;
  c.engine = cells ? NF_ENGINE_CELLS : NF_ENGINE_FOOTPRINT;
  if (cells) {
    c.fp_edge = 0.0;
    c.fp_fine = 0;
  }
  if (n_out) *n_out = total;
  return NF_OK;
}

// Crossing lists where they are the faster way: home cells run a cell's work on
// one wave, which leaves the chip idle on small packings, and evaluate every
// candidate in FP64 in full; the lists pay an atomic per rod and cell entered.
// Whole calls, home cells against lists, in us (rods in thousands):
//   one length, FP32, at 0.5 / 1 / 2 / 3 rods per excluded volume
//     20   281 276 296 448    222 232 251 276      200   372 438 495 646     428 472 542 588
//     40   292 292 288 457    283 302 325 391      400   475 533 702 937     515 583 699 829
//     60   311 310 312 472    310 347 379 411      600   583 687 805 1109    598 708 934 1114
//     100  313 324 332 499    361 399 441 495      4000  2.2 3.0 3.7 5.6 ms  2.7 3.3 4.8 6.0
//   log-normal lengths, FP32
//     60   354 452 532 368    324 355 393 408      1500  1.1 1.5 2.0 2.3 ms  1.2 1.45 1.9 2.3
//     100  365 454 554 387    359 393 447 484      2500  1.6 2.3 3.1 3.7     1.9 2.5 3.2 4.0
//     400  543 720 903 872    542 609 702 799      4000  2.4 3.4 4.6 5.8     2.9 3.5 4.7 5.6
//   one length, FP64
//     60   318 336 386 622    313 343 381 407      400   558 748 1202 1872   506 573 679 804
//     100  321 397 517 831    352 390 449 483      1000  910 1463 2516 3942  770 959 1302 1649
//     200  419 559 761 1184   419 467 534 584      8000  5.6 10.1 18.4 ms    5.2 6.6 9.7
//   log-normal lengths, FP64
//     100  356 531 724 628    360 390 437 489      8000  6.0 10.2 16.7 ms    5.6 7.0 9.5
// At a quarter and less, home cells from 80,000 rods on in all of them; at 2.4,
// FP32, one length, 100,000 and 400,000 rods 521 and 1000 against 531 and 930.
// A home cell in a dense place holds one wave up, or has to be done again in
// parts: of 16 agglomerates with peak 3 (2.8 over the mean) both ways are within
// 6 % where these lines differ from the uniform ones, with peaks 8 (6.6) / 20 (16)
//   one length, FP32, 60,000 rods at 0.8 / 1.3 440 / 486, 505 / 522 against 429 /
//   451, 430 / 456; 400,000 at 1.9 / 2.4 838 / 1109, 916 / 971 against 868 / 940,
//   894 / 867; FP64, 100,000 at 0.85 587, 686 against 497, 481
//   log-normal, FP32, 200,000 at 0.42 / 0.6 709 / 701, 1795 / 2064 against 556 /
//   584, 568 / 596; 800,000 1093 / 1168, 3036 / 3644 against 1002 / 1066, 1056 /
//   1131
static bool lists_suit(const nf_handle* h, int prec) {
  const nf_params& p = h->params[h->post_inst];
  const uint32_t n = h->n_rods[h->post_inst];
  const RodMean m = rod_mean(h, h->post_inst);
  const double crowd = (double)n * excluded_volume(m.len, m.radius) / (p.box[0] * p.box[1] * p.box[2]);
  const bool mixed = p.len_law == NF_LEN_LOGNORMAL;
  if (n <= 30000u) return true;
  if (h->desc[h->post_inst].dense >= 4.0f) {
    if (n <= 60000u) return true;
    if (mixed ? crowd >= 0.4 && n <= 800000u : crowd >= (prec == NF_PREC_FP64 ? 0.8 : 2.0) && n <= 400000u) return true;
  }
  if (prec == NF_PREC_FP64)
    return n <= 60000u || crowd >= 0.95 || (crowd >= 0.48 && n >= 200000u) || (crowd >= 0.4 && mixed);
  if (mixed) return n <= 60000u || (n <= 150000u && crowd >= 0.48) || (n <= 1500000u && crowd >= 0.8);
  return (n <= 60000u && crowd < 0.75) || (n <= 500000u && crowd >= (n < 150000u ? 2.6 : 2.3));
}

int contacts_run(nf_handle* h, double gap, uint64_t* n_out, int prec, unsigned long long*) {
  if (h->opt_contact_engine == NF_ENGINE_CELLS) return contacts_pass(h, gap, n_out, prec, WAY_CELLS);
  int rc = 1;
  // (home cells or fine cells asked for by size are the footprint pass's; lists
  // that were too short for these rods at this gap or a smaller one still are)
  if (h->opt_footprint_fine == 0 && h->opt_footprint_occ == 0 && gap < h->short_gap[h->post_inst] && lists_suit(h, prec))
    rc = contacts_pass(h, gap, n_out, prec, WAY_LISTS);
  if (rc == 1) rc = contacts_pass(h, gap, n_out, prec, WAY_SEG);
  if (rc == 1) rc = contacts_pass(h, gap, n_out, prec, WAY_CELLS);
  return rc;
}

}  // namespace nf

extern "C" int nf_contacts(nf_handle* h, double gap, uint64_t* n_contacts) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  h->err.clear();
  if (!(gap >= 0.0)) return fail(h, NF_E_INVALID, "gap must be >= 0");
  const int prec = h->opt_contact_prec >= 0 ? h->opt_contact_prec : h->params[h->post_inst].precision;
  return contacts_run(h, gap, n_contacts, prec, nullptr);
}

extern "C" int nf_get_contacts(nf_handle* h, uint32_t* row_ptr, uint32_t* col, float* gap,
                               int32_t* image, uint64_t cap) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  ContactBuffers& c = h->cb;
  if (!c.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if ((col || gap || image) && cap < c.n_contacts) return fail(h, NF_E_CAPACITY, "contact buffer too small");
  const size_t nc = c.n_contacts;
  const HostPart parts[4] = {{row_ptr, c.rowptr, row_ptr ? sizeof(uint32_t) * ((size_t)c.n_rods + 1) : 0},
                             {col, c.J, col ? sizeof(uint32_t) * nc : 0},
                             {gap, c.gap, gap ? sizeof(float) * nc : 0},
                             {image, c.img, image ? sizeof(int32_t) * nc : 0}};
  HIPCHK(h, results_to_host(h, parts, 4));
  return NF_OK;
}

extern "C" int nf_get_contact_gap64(nf_handle* h, double* gap64, uint64_t cap) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  ContactBuffers& c = h->cb;
  if (!c.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if (cap < c.n_contacts) return fail(h, NF_E_CAPACITY, "buffer too small");
  const HostPart part = {gap64, c.gap64, gap64 ? sizeof(double) * c.n_contacts : 0};
  HIPCHK(h, results_to_host(h, &part, 1));
  return NF_OK;
}

extern "C" int nf_get_contact_area(nf_handle* h, double* area, uint64_t cap) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  ContactBuffers& c = h->cb;
  if (!c.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if (cap < c.n_contacts) return fail(h, NF_E_CAPACITY, "buffer too small");
  const HostPart part = {area, c.area, area ? sizeof(double) * c.n_contacts : 0};
  HIPCHK(h, results_to_host(h, &part, 1));
  return NF_OK;
}

extern "C" int nf_contacts_stats(nf_handle* h, uint64_t* pair_tests, uint64_t* rechecks,
                                 double* max_dd, float* kernel_ms, uint64_t* tile_bytes) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  if (!h->cb.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if (pair_tests) *pair_tests = h->cb_stats[0];
  if (rechecks) *rechecks = h->cb_stats[1];
  if (max_dd) {
    const unsigned long long b = h->cb_stats[2];
    double v;
    std::memcpy(&v, &b, sizeof(v));
    *max_dd = v;
  }
  if (kernel_ms)
    for (int k = 0; k < 4; ++k) kernel_ms[k] = h->cb_ms[k];
  if (tile_bytes) *tile_bytes = h->cb_stats[3];
  return NF_OK;
}

extern "C" int nf_contacts_engine(nf_handle* h, int* engine, double* home_edge, int* fine,
                                  uint64_t* split_units) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  if (!h->cb.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if (engine) *engine = h->cb.engine;
  if (home_edge) *home_edge = h->cb.fp_edge;
  if (fine) *fine = h->cb.fp_fine;
  if (split_units) *split_units = h->cb.engine == NF_ENGINE_FOOTPRINT ? h->cb_stats[5] : 0;
  return NF_OK;
}

// ===========================================================================
// histograms
// ===========================================================================
namespace nf {

int hist_prepare(nf_handle* h, const nf_hist_spec* spec, bool want_mutual, bool want_2d,
                 double* edges, HistPlan* plan) {
  if (!h || !spec) return fail(h, NF_E_INVALID, "null argument");
  const int nb = spec->bins, npb = spec->phi_bins, ntb = spec->theta_bins;
  if (nb < 1 || nb > HIST_BINS_MAX) return fail(h, NF_E_INVALID, "bins must be 1..256");
  if (spec->centre_axis < 0 || spec->centre_axis > 2) return fail(h, NF_E_INVALID, "centre_axis must be 0..2");
  const bool two_d = npb > 0 && want_2d;
  if (two_d && (npb % 2 != 0 || ntb < 1 || npb * ntb > HIST_2D_MAX))
    return fail(h, NF_E_INVALID, "phi-theta needs even phi_bins and phi*theta <= 4096");
  if (want_mutual && !h->cb.valid) return fail(h, NF_E_STATE, "mutual-angle histogram needs nf_contacts first");
  const double PI = 3.14159265358979323846;
  // edges: polar [nb+1], mutual [nb+1], then theta [ntb+1] and phi [half+1]
  size_t k0 = 0;
  for (int k = 0; k <= nb; ++k) edges[k0 + k] = std::cos((double)k * PI / (double)nb);
  k0 += (size_t)nb + 1;
  for (int k = 0; k <= nb; ++k) edges[k0 + k] = std::cos((double)k * (0.5 * PI) / (double)nb);
  k0 += (size_t)nb + 1;
  if (two_d) {
    const int half = npb / 2;
    for (int k = 0; k <= ntb; ++k) edges[k0 + k] = std::cos((double)k * PI / (double)ntb);
    k0 += (size_t)ntb + 1;
    for (int k = 0; k <= half; ++k) edges[k0 + k] = std::cos((double)k * PI / (double)half);
    k0 += (size_t)half + 1;
  }
  double mu[3] = {spec->pol_axis[0], spec->pol_axis[1], spec->pol_axis[2]};
  const double mn = std::sqrt((mu[0] * mu[0] + mu[1] * mu[1]) + mu[2] * mu[2]);
  if (!(mn > 0.0)) return fail(h, NF_E_INVALID, "pol_axis must be non-zero");
  for (int k = 0; k < 3; ++k) plan->mu[k] = mu[k] / mn;
  plan->nb = nb;
  plan->npb = two_d ? npb : 0;
  plan->ntb = two_d ? ntb : 0;
  plan->axis = spec->centre_axis;
  plan->mutual = want_mutual;
  plan->n_edges = k0;
  plan->n_out = 3 * (size_t)nb + (two_d ? (size_t)npb * ntb : 0);
  return NF_OK;
}

int hist_run(nf_handle* h, const HistPlan& pl, const double* edges, double* dE,
             unsigned long long* dOut, int64_t* out_centre, int64_t* out_polar, int64_t* out_mutual,
             int64_t* out_phitheta, bool may_allocate) {
  hipStream_t s = h->stream;
  const int nb = pl.nb;
  hipError_t e = hipMemcpyAsync(dE, edges, sizeof(double) * pl.n_edges, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) {
    fill_u32((uint32_t*)dOut, 0u, 2 * pl.n_out, s);
    e = hipGetLastError();
  }
  const InstDesc& d = h->desc[h->post_inst];
  const uint32_t n = h->n_rods[h->post_inst];
  if (e == hipSuccess && n) {
    launch_hist(h->gb.bP + d.rod_off, h->gb.bD + d.rod_off, n, pl.mutual ? h->cb.n_contacts : 0, h->cb.I,
                h->cb.J, dE, dE + (nb + 1), pl.npb ? dE + 2 * (nb + 1) : nullptr, nb, pl.npb, pl.ntb,
                pl.axis, h->params[h->post_inst].box[pl.axis], pl.mu, dOut, s);
    e = hipGetLastError();
  }
  // int64 and u64 share the layout; counts never reach 2^63
  const int64_t* src = (const int64_t*)dOut;
  auto part = [&](int64_t* dst, size_t off, size_t len) {
    return HostPart{dst, src + off, dst ? sizeof(int64_t) * len : 0};
  };
  const HostPart parts[4] = {part(out_centre, 0, nb), part(out_polar, nb, nb),
                             part(pl.mutual ? out_mutual : nullptr, 2 * (size_t)nb, nb),
                             part(pl.npb ? out_phitheta : nullptr, 3 * (size_t)nb, (size_t)pl.npb * pl.ntb)};
  hipError_t w = hipSuccess;
  if (may_allocate || h->pin) {
    w = to_host(h, parts, 4);  // (waits for the upload of `edges` too)
  } else {
    for (const HostPart& q : parts)
      if (w == hipSuccess && q.bytes) w = hipMemcpyAsync(q.dst, q.src, q.bytes, hipMemcpyDeviceToHost, s);
    const hipError_t sy = sync_stream(s, "histograms");
    if (w == hipSuccess) w = sy;
  }
  if (e == hipSuccess) e = w;
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("histograms: ") + hipGetErrorString(e));
  return NF_OK;
}

}  // namespace nf

extern "C" int nf_histograms(nf_handle* h, const nf_hist_spec* spec, int64_t* out_centre,
                             int64_t* out_polar, int64_t* out_mutual, int64_t* out_phitheta) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  double edges[HIST_EDGES_MAX];
  HistPlan pl;
  int rc = hist_prepare(h, spec, out_mutual != nullptr, out_phitheta != nullptr, edges, &pl);
  if (rc != NF_OK) return rc;
  double* dE = nullptr;
  unsigned long long* dOut = nullptr;
  rc = dalloc(h, &dE, pl.n_edges);
  if (rc == NF_OK) rc = dalloc(h, &dOut, pl.n_out);
  if (rc == NF_OK)
    rc = hist_run(h, pl, edges, dE, dOut, out_centre, out_polar, out_mutual, out_phitheta, true);
  dfree(h, dE);
  dfree(h, dOut);
  return rc;
}

// Centre-centre distance statistics of instance 0 (statKernel_CENT via
// collectStats, src/statistics_collection.cu:866-1033).
extern "C" int nf_centre_distance(nf_handle* h, int32_t bins, double width, int64_t* counts,
                                  uint64_t* n_pairs, uint64_t* sum_d_q24, uint64_t* sum_d2_q16) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  if (bins < 1 || bins > CENT_BINS_MAX || !(width > 0.0))
    return fail(h, NF_E_INVALID, "need 1 <= bins <= 1024 and width > 0");
  const nf_params& p = h->params[h->post_inst];
  const uint32_t n = h->n_rods[h->post_inst];
  const double rmax = bins * width;
  const double bmin = std::min(p.box[0], std::min(p.box[1], p.box[2]));
  if (rmax > 8.0 * bmin) return fail(h, NF_E_INVALID, "bins * width exceeds 8 box edges");
  hipStream_t s = h->stream;
  const float4* P = h->gb.bP + h->desc[h->post_inst].rod_off;
  const float4* D = h->gb.bD + h->desc[h->post_inst].rod_off;
  const double density = (double)n / (p.box[0] * p.box[1] * p.box[2]);
  int32_t nc[3];
  auto cells_of = [&](double edge) {
    uint64_t c = 1;
    for (int a = 0; a < 3; ++a) {
      nc[a] = (int32_t)std::min(std::max(std::floor(p.box[a] / edge), 1.0), 1024.0);
      c *= (uint64_t)nc[a];
    }
    return c;
  };
  if (cells_of(default_cell_edge(rmax, density, 1.0)) > (1ull << 26))
    return fail(h, NF_E_INVALID, "statistics grid too large");
  std::vector<double> e2(bins + 1);
  for (int k = 0; k <= bins; ++k) e2[k] = ((double)k * width) * ((double)k * width);
  float4* cP = nullptr;
  float4* cD = nullptr;
  uint32_t *cid = nullptr, *cstart = nullptr, *ccount = nullptr, *cells = nullptr;
  float* chl = nullptr;
  int4* dst = nullptr;
  double* de2 = nullptr;
  unsigned long long *out = nullptr, *part = nullptr;
  int rc = NF_OK;
  const uint64_t n1 = std::max<uint64_t>(n, 1);
  BinScratch bs;
  std::vector<int4> runs;
  uint64_t ncells = 0;
  auto release_grid = [&]() {
    void* w[] = {cstart, ccount, chl, dst};
    for (void* q : w) dfree(h, q);
    free_bin_scratch(h, &bs);
    cstart = ccount = nullptr;
    chl = nullptr;
    dst = nullptr;
  };
  // the rods on cells of `edge`, and the half stencil as runs of cells along x
  auto layout = [&](double edge) -> int {
    release_grid();
    ncells = cells_of(edge);
    double scale[3];
    for (int a = 0; a < 3; ++a) scale[a] = (double)nc[a] / p.box[a];
    std::vector<int4> st = build_stencil(nc, p.box, rmax, true);
    std::sort(st.begin(), st.end(), [](const int4& a, const int4& b) {
      return a.z != b.z ? a.z < b.z : (a.y != b.y ? a.y < b.y : a.x < b.x);
    });
    runs.clear();
    for (const int4& o : st) {
      if (!runs.empty() && runs.back().z == o.y && runs.back().w == o.z && runs.back().y + 1 == o.x)
        runs.back().y = o.x;
      else
        runs.push_back(make_int4(o.x, o.x, o.y, o.z));
    }
    int r = dalloc(h, &cstart, ncells + 1);
    if (r == NF_OK) r = dalloc(h, &ccount, ncells);
    if (r == NF_OK) r = dalloc(h, &chl, ncells);
    if (r == NF_OK) r = dalloc(h, &dst, runs.size());
    if (r != NF_OK) return r;
    const hipError_t u = hipMemcpyAsync(dst, runs.data(), sizeof(int4) * runs.size(), hipMemcpyHostToDevice, s);
    if (u != hipSuccess) return fail(h, NF_E_HIP, std::string("statistics upload: ") + hipGetErrorString(u));
    return bin_rods(h, P, D, n, nc, scale, cP, cD, cid, cstart, ccount, chl, &bs);
  };
  if (rc == NF_OK) rc = dalloc(h, &cP, n1);
  if (rc == NF_OK) rc = dalloc(h, &cD, n1);
  if (rc == NF_OK) rc = dalloc(h, &cid, n1);
  if (rc == NF_OK) rc = dalloc(h, &part, (size_t)CENT_BLOCKS * (bins + 3));
  if (rc == NF_OK) rc = dalloc(h, &de2, (size_t)bins + 1);
  if (rc == NF_OK) rc = dalloc(h, &out, (size_t)bins + 3);
  auto release = [&]() {
    (void)sync_stream(s, "centre distance");
    release_grid();
    void* w[] = {cP, cD, cid, cells, de2, part, out};
    for (void* q : w) dfree(h, q);
  };
  if (rc != NF_OK) {
    release();
    return rc;
  }
  hipError_t e = hipMemcpyAsync(de2, e2.data(), sizeof(double) * e2.size(), hipMemcpyHostToDevice, s);
  if (e != hipSuccess) {
    release();
    return fail(h, NF_E_HIP, std::string("statistics upload: ") + hipGetErrorString(e));
  }
  // grid: edge just over rmax and the stencil's margin (half stencil of +-1
  // cells; at rmax itself a box of whole edges has cells two away in it, three
  // times the candidates), finer when crowded.  Where that makes many cells,
  // wide enough for 16 rods a cell, so that a run of three fills a wave's 64
  // lanes: 300,000 rods within 0.05 um of each other 29 ms on cells of that edge
  // (most of them empty), with 4, 8, 16, 24 rods a cell 0.27, 0.20, 0.155, 0.175
  // ms; 1M rods within 0.13 um 6.9 and 0.78, 0.53, 0.39, 0.44 ms.  17,500 cells
  // for 2,000 rods take 80 us, with the look at their crowding below 75-98;
  // 23,000 for 20,000 rods 110, 97-111.
  const double near_edge = default_cell_edge(rmax + 1.01 * (double)CELL_MARGIN, density, 1.0);
  double edge = near_edge;
  if (density > 0.0 && cells_of(near_edge) > 16384) edge = std::max(near_edge, std::cbrt(16.0 / density));
  rc = layout(edge);
  double mean = (double)n / (double)std::max<uint64_t>(ncells, 1);  // rods in a cell that holds any
  if (rc == NF_OK && edge > near_edge) {
    // Widened cells suit rods that are spread out: where a rod shares its cell
    // with four times the others that it would in an even packing (agglomerates
    // three times as dense as the mean reach two), cells for 16 of the rods as
    // they lie, and the empty ones, most then, are left out by a list.
    HostScalars* scalars = host_scalars(h);
    fill_u32((uint32_t*)out, 0u, 2, s);
    launch_cent_crowd(ccount, ncells, out, s);
    e = scalars_to_host(h, scalars->ctr, out, sizeof(unsigned long long));
    if (e == hipSuccess) e = sync_stream(s, "centre distance");
    const double crowd = (double)scalars->ctr[0] / (double)n1;
    if (e == hipSuccess && crowd > 4.0 * (mean + 1.0)) {
      const double cell = p.box[0] * p.box[1] * p.box[2] / (double)ncells;
      rc = layout(std::max(near_edge, std::cbrt(16.0 * cell / crowd)));
      mean = std::max(16.0, crowd * p.box[0] * p.box[1] * p.box[2] / (double)ncells / cell);
      if (rc == NF_OK) rc = dalloc(h, &cells, std::min<uint64_t>(n1, ncells) + 1);
      if (rc == NF_OK) launch_cent_cells(ccount, ncells, cells, s);
    }
  }
  if (rc != NF_OK || e != hipSuccess) {
    release();
    return rc != NF_OK ? rc : fail(h, NF_E_HIP, std::string("centre distance: ") + hipGetErrorString(e));
  }
  fill_u32((uint32_t*)out, 0u, 2 * ((uint64_t)bins + 3), s);
  const double Lmax = std::max(p.box[0], std::max(p.box[1], p.box[2]));
  const float ew = (float)(5.9604644775390625e-8 * (Lmax + rmax) * 1.01);
  const float rf = (float)rmax + 8.0f * ew;
  launch_cent(cP, cid, cstart, ccount, cells, dst, (uint32_t)runs.size(), mean, nc, p.box, de2, bins, width,
              rf * rf * 1.00001f, part, out, s);
  std::vector<unsigned long long> hout((size_t)bins + 3);
  const HostPart out_part = {hout.data(), out, sizeof(unsigned long long) * hout.size()};
  e = to_host(h, &out_part, 1);
  if (e == hipSuccess) e = hipGetLastError();
  release();
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("centre distance: ") + hipGetErrorString(e));
  if (counts)
    for (int k = 0; k < bins; ++k) counts[k] = (int64_t)hout[k];
  if (n_pairs) *n_pairs = hout[bins];
  if (sum_d_q24) *sum_d_q24 = hout[bins + 1];
  if (sum_d2_q16) *sum_d2_q16 = hout[bins + 2];
  return NF_OK;
}

// Van der Waals energy over the contacts of the last nf_contacts call
// (collect_vdw, src/statistics_collection.cu:53-154).
extern "C" int nf_vdw(nf_handle* h, double A, double B, double* energy, uint64_t* n_pairs) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  ContactBuffers& c = h->cb;
  if (!c.valid) return fail(h, NF_E_STATE, "no contacts computed");
  if (!(c.gap_cut > 0.0)) return fail(h, NF_E_INVALID, "the contact gap must be > 0");
  hipStream_t s = h->stream;
  const uint32_t n = c.n_rods;
  const float4* P = h->gb.bP + h->desc[h->post_inst].rod_off;
  const float4* D = h->gb.bD + h->desc[h->post_inst].rod_off;
  double *rowsum = nullptr, *bsum = nullptr, *tot = nullptr;
  unsigned long long* pairs = nullptr;
  int rc = NF_OK;
  const uint64_t nb = ((uint64_t)n + 1023) / 1024;
  if (rc == NF_OK) rc = dalloc(h, &rowsum, std::max<uint64_t>(n, 1));
  if (rc == NF_OK) rc = dalloc(h, &bsum, std::max<uint64_t>(nb, 1));
  if (rc == NF_OK) rc = dalloc(h, &tot, 1);
  if (rc == NF_OK) rc = dalloc(h, &pairs, 1);
  auto release = [&]() {
    dfree(h, rowsum);
    dfree(h, bsum);
    dfree(h, tot);
    dfree(h, pairs);
  };
  if (rc != NF_OK) {
    release();
    return rc;
  }
  fill_u32((uint32_t*)pairs, 0u, 2, s);
  launch_vdw(P, D, n, c.rowptr, c.J, c.img, h->params[h->post_inst].box, c.gap_cut, A, B, rowsum, bsum, tot,
             pairs, s);
  double e_h = 0.0;
  unsigned long long p_h = 0;
  hipError_t e = hipMemcpyAsync(&e_h, tot, sizeof(double), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipMemcpyAsync(&p_h, pairs, sizeof(p_h), hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = sync_stream(s, "van der Waals");
  if (e == hipSuccess) e = hipGetLastError();
  release();
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("van der Waals: ") + hipGetErrorString(e));
  if (energy) *energy = e_h;
  if (n_pairs) *n_pairs = p_h;
  return NF_OK;
}
