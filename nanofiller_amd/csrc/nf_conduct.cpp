// nf_conduct.cpp - host side of the DC conductance solve on the network of
// the last nf_network call (see nf_solve.hip): reduced system, conjugate
// gradients with a convergence check every CG_CHECK iterations, currents and
// rod potentials.  The check itself runs on the device; on a long solve the
// next iterations are queued before its verdict is read, and do nothing if it
// was the last.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <cmath>
#include <string>
#include <vector>

#include "nf_host.h"

using namespace nf;

namespace {
constexpr uint32_t CG_CHECK = 16;  // iterations between convergence checks
// Iterations from which one batch is queued ahead: a converged solve then has
// 32 launches that do nothing (60 us), against 8 us of waiting per check.
constexpr uint32_t CG_AHEAD = 128;
}

extern "C" int nf_conductance(nf_handle* h, double tol, uint32_t max_iter, nf_conductance_info* info,
                              double* potentials) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  ContactBuffers& c = h->cb;
  if (!c.net_valid) return fail(h, NF_E_STATE, "no network built (call nf_network first)");
  if (!(tol > 0.0) || max_iter == 0) return fail(h, NF_E_INVALID, "tol must be > 0 and max_iter > 0");
  const uint32_t n = c.n_rods;
  hipStream_t s = h->stream;
  uint32_t *flag = nullptr, *act = nullptr, *rl = nullptr, *idx = nullptr, *off = nullptr,
           *tmp = nullptr, *crow = nullptr, *ccol = nullptr;
  double *cval = nullptr, *dinv = nullptr, *bsrc = nullptr, *bsnk = nullptr, *x = nullptr,
         *r = nullptr, *pv = nullptr, *q = nullptr, *part = nullptr, *vdev = nullptr;
  double2* zp = nullptr;
  CgScal *scal = nullptr, *verdicts = nullptr;
  uint32_t *acto = nullptr, *rlo = nullptr, *idxo = nullptr, *offo = nullptr;
  auto release = [&]() {
    void* ptrs[] = {flag, act, rl,   idx, off, tmp,  crow, ccol, cval, dinv, bsrc, bsnk,
                    x,    r,   zp,   pv,  q,   part, vdev, scal, acto, rlo,  idxo, offo, verdicts};
    for (void* p : ptrs) dfree(h, p);
  };
  const uint64_t n1 = (uint64_t)n + 1;
  int rc = NF_OK;
#define ALLOC(ptr, cnt) \
  if (rc == NF_OK) rc = dalloc(h, &(ptr), (size_t)std::max<uint64_t>((cnt), 1));
  ALLOC(flag, n);
  ALLOC(act, n1);
  ALLOC(rl, n1);
  ALLOC(idx, n1);
  ALLOC(off, n1);
  ALLOC(tmp, scan_tmp_words(n1));
  ALLOC(part, 3 * CG_MAX_BLOCKS);
  ALLOC(scal, 1);
  if (rc != NF_OK) {
    release();
    return rc;
  }
  // reduced system: rods of the components touching both electrodes
  fill_u32(flag, 0u, std::max<uint64_t>(n, 1), s);
  fill_u32(act, 0u, n1, s);
  fill_u32(rl, 0u, n1, s);
  if (n > 0) {
    launch_cs_flag(c.nrow, c.ncol, c.labels, n, flag, s);
    launch_cs_active(c.nrow, c.ncol, c.labels, flag, n, act, rl, s);
  }
  // unknowns numbered in the cell list's (spatial) order when the packing's
  // cell list is at hand, else in rod order
  const bool spatial = c.cid != nullptr && c.cell_list != 0 && n > 0;
  if (spatial) {
    if (rc == NF_OK) rc = dalloc(h, &acto, n1);
    if (rc == NF_OK) rc = dalloc(h, &rlo, n1);
    if (rc == NF_OK) rc = dalloc(h, &idxo, n1);
    if (rc == NF_OK) rc = dalloc(h, &offo, n1);
    if (rc != NF_OK) {
      release();
      return rc;
    }
    fill_u32(acto + n, 0u, 1, s);
    fill_u32(rlo + n, 0u, 1, s);
    launch_cs_order(n, c.cid, act, rl, acto, rlo, nullptr, nullptr, nullptr, nullptr, 0, s);
    scan_u32(acto, idxo, n1, tmp, s);
    scan_u32(rlo, offo, n1, tmp, s);
    launch_cs_order(n, c.cid, nullptr, nullptr, nullptr, nullptr, idxo, offo, idx, off, 1, s);
  } else {
    scan_u32(act, idx, n1, tmp, s);
    scan_u32(rl, off, n1, tmp, s);
  }
  uint32_t mn[2] = {0, 0};
  if (hipError_t e_ = hipMemcpyAsync(&mn[0], idx + n, sizeof(uint32_t), hipMemcpyDeviceToHost, s); e_ != hipSuccess) {
      release();
      return fail(h, NF_E_HIP, std::string("conductance copy: ") + hipGetErrorString(e_));
    }
  if (hipError_t e_ = hipMemcpyAsync(&mn[1], off + n, sizeof(uint32_t), hipMemcpyDeviceToHost, s); e_ != hipSuccess) {
      release();
      return fail(h, NF_E_HIP, std::string("conductance copy: ") + hipGetErrorString(e_));
    }
  if (hipError_t e = sync_stream(s, "conductance set-up"); e != hipSuccess) {
    release();
    return fail(h, NF_E_HIP, std::string("conductance set-up: ") + hipGetErrorString(e));
  }
  {
    void* q[] = {acto, rlo, idxo, offo};
    for (void* p : q) dfree(h, p);
    acto = rlo = idxo = offo = nullptr;
  }
  const uint32_t m = mn[0], nnz = mn[1];
  nf_conductance_info out{};
  out.unknowns = m;
  out.converged = 1;
  float solve_ms = 0.0f;
  if (m > 0) {
    ALLOC(crow, (uint64_t)m + 1);
    ALLOC(ccol, nnz);
    ALLOC(cval, nnz);
    ALLOC(dinv, m);
    ALLOC(bsrc, m);
    ALLOC(bsnk, m);
    ALLOC(x, m);
    ALLOC(r, m);
    ALLOC(zp, m);
    ALLOC(pv, m);
    ALLOC(q, m);
    if (rc != NF_OK) {
      release();
      return rc;
    }
    HostScalars* scalars = host_scalars(h);
    if (!h->scal_pinned) {
      ALLOC(verdicts, 2);
      if (rc != NF_OK) {
        release();
        return rc;
      }
    }
    launch_cs_fill(c.nrow, c.ncol, c.nval, n, act, idx, off, crow, ccol, cval, dinv, bsrc, bsnk, s);
    fill_u32(crow + m, nnz, 1, s);
    CgArgs a{m, 0, 0, crow, ccol, cval, dinv, bsrc, bsnk, x, r, pv, q, zp,
             part, part + CG_MAX_BLOCKS, part + 2 * CG_MAX_BLOCKS, scal};
    cg_grids(a);
    struct Check {
      uint32_t it;     // iterations before it
      CgScal* host;    // copy of the scalars on the host
      CgScal* out;     // where the kernel leaves it: there, or in device memory if the host has none pinned
      hipEvent_t done;
    };
    CgScal* out0 = h->scal_pinned ? scalars->cg : verdicts;
    Check slot[2] = {{0, &scalars->cg[0], out0, h->ev[2]}, {0, &scalars->cg[1], out0 + 1, h->ev[3]}};
    auto fetch = [&](const Check& c) -> hipError_t {
      return c.out == c.host ? hipSuccess : scalars_to_host(h, c.host, c.out, sizeof(CgScal));
    };
    uint32_t pending = 0, newest = 0;
    hipEventRecord(h->ev[0], s);
    // queues what leads to the next check (init for the first) and the check, which leaves its verdict in c.host
    auto queue = [&](uint32_t it, uint32_t count, Check& c) -> hipError_t {
      if (count == 0)
        launch_cg_init(a, tol, c.out, s);
      else
        launch_cg_iterations(a, it, count, tol, c.out, s);
      c.it = it + count;
      ++pending;
      const hipError_t e = fetch(c);
      return e == hipSuccess ? hipEventRecord(c.done, s) : e;
    };
    uint32_t it = 0;
    CgScal hs{};
    hipError_t e = queue(0, 0, slot[0]);
    for (;;) {
      Check& oldest = slot[newest ^ (pending - 1u)];
      const uint32_t last = slot[newest].it;
      if (e == hipSuccess && pending == 1 && last >= CG_AHEAD && last < max_iter) {
        newest ^= 1u;
        e = queue(last, std::min(CG_CHECK, max_iter - last), slot[newest]);
      }
      if (e == hipSuccess) e = sync_event(oldest.done, "conductance iterations");
      if (e != hipSuccess) {
        release();
        return fail(h, NF_E_HIP, std::string("conductance iterations: ") + hipGetErrorString(e));
      }
      --pending;
      hs = *oldest.host;
      it = oldest.it;
      out.residual = hs.res;
      if (hs.done || it >= max_iter) break;
      if (pending == 0) {
        newest ^= 1u;
        e = queue(it, std::min(CG_CHECK, max_iter - it), slot[newest]);
      }
    }
    const bool conv = hs.done == CG_CONVERGED;
    launch_cg_current(a, slot[0].out, s);  // (after whatever is queued: both slots are free by then)
    hipEventRecord(h->ev[1], s);
    e = fetch(slot[0]);
    if (e == hipSuccess) e = sync_stream(s, "conductance currents");
    if (e != hipSuccess) {
      release();
      return fail(h, NF_E_HIP, std::string("conductance currents: ") + hipGetErrorString(e));
    }
    hs = scalars->cg[0];
    hipEventElapsedTime(&solve_ms, h->ev[0], h->ev[1]);
    out.iterations = it;
    out.converged = conv ? 1 : 0;
    out.conductance = hs.isrc;
    out.current_sink = hs.isnk;
  }
  out.solve_ms = solve_ms;
  if (potentials && n > 0) {
    ALLOC(vdev, n);
    if (rc != NF_OK) {
      release();
      return rc;
    }
    launch_cs_potential(n, c.labels, flag, act, idx, x, vdev, s);
    const HostPart part = {potentials, vdev, sizeof(double) * n};
    if (hipError_t e = to_host(h, &part, 1); e != hipSuccess) {
      release();
      return fail(h, NF_E_HIP, std::string("conductance potentials: ") + hipGetErrorString(e));
    }
  }
#undef ALLOC
  release();
  if (info) *info = out;
  return NF_OK;
}
