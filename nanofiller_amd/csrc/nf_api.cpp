// nf_api.cpp - C ABI of the library: parameter normalisation, handle
// lifecycle, batched generation (HIP-graph rounds), contacts, histograms,
// copies out.  Host orchestration only; all per-rod and per-pair work runs
// in the HIP kernels of nf_gen.hip, nf_pair.hip and nf_post.hip.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <array>
#include <chrono>
#include <cmath>
#include <cstdarg>
#include <cstdlib>
#include <thread>
#include <cstdio>
#include <cstring>
#include <string>
#include <vector>

#include "nf_internal.h"
#include "nf_host.h"

using namespace nf;

std::string g_last_error;

namespace nf {

int fail(nf_handle* h, int code, const std::string& msg) {
  if (h)
    h->err = msg;
  else
    g_last_error = msg;
  return code;
}

// Size classes: 256 B granules below 64 KiB, then four classes per power of
// two, so a reused block wastes at most a quarter of its size.
static size_t size_class(size_t bytes) {
  if (bytes <= 65536) return (bytes + 255) & ~(size_t)255;
  size_t p = 65536;
  while (p < bytes) p <<= 1;
  const size_t q = p >> 3;  // p/2 + k*p/8, k = 1..4
  size_t c = p >> 1;
  while (c < bytes) c += q;
  return c;
}

constexpr size_t POOL_CAP = (size_t)16 << 30;  // freed bytes kept per handle

constexpr size_t SLAB_FROM = (size_t)1 << 20, SLAB_TO = (size_t)32 << 20, SLAB_LARGEST = (size_t)256 << 20;

constexpr size_t SMALL_TO = (size_t)128 << 10, SMALL_SLAB = (size_t)1 << 20;

static nf_handle::Slab* slab_of(nf_handle* h, const void* p) {
  for (auto& kind : h->slabs)
    for (auto& s : kind)
      if ((const char*)p >= s.p && (const char*)p < s.p + s.size) return &s;
  return nullptr;
}

// Takes the blocks of a slab without one in use out of the pool.
static void clear_slab(nf_handle* h, nf_handle::Slab& s) {
  for (auto it = h->pool.begin(); it != h->pool.end();) {
    if ((char*)it->second < s.p || (char*)it->second >= s.p + s.size) {
      ++it;
      continue;
    }
    h->pool_bytes -= it->first;
    it = h->pool.erase(it);
  }
  s.used = 0;
}

// A block cut from the newest slab, from one whose blocks are all free, or
// from a new one (of large blocks twice the newest's size); null if there is no
// memory for one.
static void* slab_block(nf_handle* h, size_t cls) {
  const bool small = cls <= SMALL_TO;
  auto& slabs = h->slabs[small ? 0 : 1];
  if (slabs.empty() || slabs.back().size - slabs.back().used < cls) {
    auto idle =
        std::find_if(slabs.begin(), slabs.end(), [&](const nf_handle::Slab& s) { return s.live == 0 && s.size >= cls; });
    if (idle != slabs.end()) {
      clear_slab(h, *idle);
      std::rotate(idle, idle + 1, slabs.end());
    } else {
      const size_t size = small ? SMALL_SLAB : (slabs.empty() ? SLAB_TO : std::min(2 * slabs.back().size, SLAB_LARGEST));
      void* p = nullptr;
      if (hipMalloc(&p, size) != hipSuccess) {
        (void)hipGetLastError();
        return nullptr;
      }
      slabs.push_back({(char*)p, size, 0, 0});
    }
  }
  auto& s = slabs.back();
  void* q = s.p + s.used;
  s.used += cls;
  return q;
}

// Gives the pool's blocks back to the device: those of their own, and the
// slabs without a block in use.
static void trim_pool(nf_handle* h) {
  for (auto& slabs : h->slabs)
    for (size_t k = 0; k < slabs.size();) {
      if (slabs[k].live != 0) {
        ++k;
        continue;
      }
      clear_slab(h, slabs[k]);
      (void)hipFree(slabs[k].p);
      slabs.erase(slabs.begin() + k);
    }
  for (auto it = h->pool.begin(); it != h->pool.end();) {
    if (slab_of(h, it->second)) {
      ++it;
      continue;
    }
    (void)hipFree(it->second);
    h->pool_bytes -= it->first;
    it = h->pool.erase(it);
  }
}

static bool shed_lists(nf_handle* h);

int dalloc_bytes(nf_handle* h, void** p, size_t bytes) {
  *p = nullptr;
  if (bytes == 0) bytes = 16;
  const size_t cls = size_class(bytes);
  auto it = h->pool.find(cls);
  void* q = nullptr;
  if (it != h->pool.end()) {
    q = it->second;
    h->pool.erase(it);
    h->pool_bytes -= cls;
  } else {
    if (cls <= SMALL_TO || (cls >= SLAB_FROM && cls <= SLAB_TO)) q = slab_block(h, cls);
    hipError_t e = q ? hipSuccess : hipMalloc(&q, cls);
    if (e != hipSuccess) {
      // give the cached blocks back and try once more
      (void)hipGetLastError();
      trim_pool(h);
      e = hipMalloc(&q, cls);
    }
    if (e != hipSuccess && shed_lists(h)) {
      (void)hipGetLastError();
      trim_pool(h);
      e = hipMalloc(&q, cls);
    }
    // a caller may do without the block: its next check of the runtime's last
    // error must not find this one
    if (e != hipSuccess) (void)hipGetLastError();
    if (e != hipSuccess)
      return fail(h, NF_E_NOMEM,
                  "hipMalloc of " + std::to_string(cls) + " bytes failed: " + hipGetErrorString(e));
  }
  if (auto* s = slab_of(h, q)) ++s->live;
  h->allocs[q] = cls;
  *p = q;
  return NF_OK;
}

static bool trace_on() {
  static int on = -1;
  if (on < 0) {
    const char* e = std::getenv("NF_TRACE");
    on = (e && *e && *e != '0') ? 1 : 0;
  }
  return on == 1;
}

void trace(const char* fmt, ...) {
  if (!trace_on()) return;
  va_list ap;
  va_start(ap, fmt);
  std::fprintf(stderr, "[nf] ");
  std::vfprintf(stderr, fmt, ap);
  std::fprintf(stderr, "\n");
  std::fflush(stderr);
  va_end(ap);
}

template <class Query>
static hipError_t poll(Query query, const char* what) {
  static double limit = -1.0;
  if (limit < 0.0) {
    const char* e = std::getenv("NF_SYNC_TIMEOUT_S");
    limit = e ? std::atof(e) : 120.0;
    if (!(limit > 0.0)) limit = 120.0;
  }
  const auto t0 = std::chrono::steady_clock::now();
  for (;;) {
    const hipError_t e = query();
    if (e != hipErrorNotReady) return e;
    const double el = std::chrono::duration<double>(std::chrono::steady_clock::now() - t0).count();
    if (el > limit) {
      std::fprintf(stderr, "[nf] %s: stream not done after %.0f s\n", what, el);
      std::fflush(stderr);
      return hipErrorLaunchTimeOut;
    }
    // (a sleep of 2 us lasts 60: short waits spin)
    if (el < 0.002)
      std::this_thread::yield();
    else
      std::this_thread::sleep_for(std::chrono::microseconds(el < 0.01 ? 2 : 200));
  }
}

hipError_t sync_stream(hipStream_t s, const char* what) {
  return poll([&] { return hipStreamQuery(s); }, what);
}

hipError_t sync_event(hipEvent_t ev, const char* what) {
  return poll([&] { return hipEventQuery(ev); }, what);
}

// Returns a block to the handle's pool.  The handle's stream is drained
// first (usually already idle), so no queued kernel can still use a block
// that a later call receives.
void dfree(nf_handle* h, void* p) {
  if (!p) return;
  auto it = h->allocs.find(p);
  if (it == h->allocs.end()) {
    (void)hipFree(p);
    return;
  }
  const size_t cls = it->second;
  h->allocs.erase(it);
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (auto* s = slab_of(h, p)) {
    --s->live;
  } else if (h->pool_bytes + cls > POOL_CAP) {
    (void)hipFree(p);
    return;
  }
  h->pool.emplace(cls, p);
  h->pool_bytes += cls;
}

}  // namespace nf

// ===========================================================================
// parameters
// ===========================================================================
extern "C" void nf_params_default(nf_params* p) {
  std::memset(p, 0, sizeof(*p));
  // simPrms::simPrms (src/simPrms.cpp:22-117)
  p->vol_frac = 0.05 / 100.0;
  p->len_law = NF_LEN_CONST;
  p->len = 4.0;
  p->len_sigma = 0.0;
  p->len_min = 0.0;
  p->len_max = 0.0;
  p->radius = 0.010;
  p->sep = 0.0;
  p->soft_frac = 1.0;
  p->ort_law = NF_ORT_ISO;
  p->kappa = 0.0;
  p->axis[0] = 0.0;
  p->axis[1] = 0.0;
  p->axis[2] = 1.0;
  p->den_law = NF_DEN_UNIFORM;
  p->agg_sigma = 1.0;
  p->agg_peak = 1.0;
  p->contact_gap = 0.015;
  p->max_rounds = 1000;  // cudaMain.cu:113
  p->stall_rounds = 8;
  p->min_batch = 64;
  p->max_batch = 0;
  p->cell_size = 0.0;
  p->precision = NF_PREC_FP32_RECHECK;
  p->elec_axis = 0;
  p->tunnel_lambda = 1e-4;
  p->tunnel_g0 = 1.0;
  p->seed = 1;
  p->stream = 0;
}

double nf::default_cell_edge(double reach_typ, double density, double factor) {
  double e = factor * reach_typ;
  if (density > 0.0 && density * e * e * e > 256.0) {
    e = std::cbrt(32.0 / density);
    if (e < 0.25 * reach_typ) e = 0.25 * reach_typ;
    if (e > reach_typ) e = reach_typ;
  }
  return e;
}

double nf::excluded_volume(double L, double a) {
  const double D = 2.0 * a;
  const double PI = 3.14159265358979323846;
  return 0.5 * PI * D * L * L + 2.0 * PI * D * D * L + (4.0 * PI / 3.0) * D * D * D;
}

RodMean nf::rod_mean(const nf_handle* h, int inst) {
  if (!h->generated && h->given[inst].radius > 0.0) return h->given[inst];
  return {h->params[inst].len, h->params[inst].radius};
}

extern "C" int nf_params_normalize(nf_params* p) {
  for (int d = 0; d < 3; ++d) {
    if (!(p->box[d] > 0.0)) return fail(nullptr, NF_E_INVALID, "box edges must be > 0");
    p->box[d] = (double)(float)p->box[d];
  }
  if (!(p->radius > 0.0)) return fail(nullptr, NF_E_INVALID, "radius must be > 0");
  if (!(p->len > 0.0)) return fail(nullptr, NF_E_INVALID, "length must be > 0");
  if (p->len_law == NF_LEN_LOGNORMAL) {
    if (!(p->len_min > 0.0) || !(p->len_max >= p->len_min) || !(p->len_sigma >= 0.0))
      return fail(nullptr, NF_E_INVALID, "log-normal length needs 0 < len_min <= len_max, sigma >= 0");
  } else if (p->len_law != NF_LEN_CONST) {
    return fail(nullptr, NF_E_INVALID, "unknown length law");
  }
  if (p->ort_law == NF_ORT_VMF) {
    if (!(p->kappa > 0.0)) return fail(nullptr, NF_E_INVALID, "vMF kappa must be > 0");
    const double n = std::sqrt((p->axis[0] * p->axis[0] + p->axis[1] * p->axis[1]) + p->axis[2] * p->axis[2]);
    if (!(n > 0.0)) return fail(nullptr, NF_E_INVALID, "vMF axis must be non-zero");
    for (int d = 0; d < 3; ++d) p->axis[d] = p->axis[d] / n;
  } else if (p->ort_law != NF_ORT_ISO) {
    return fail(nullptr, NF_E_INVALID, "unknown orientation law");
  }
  if (p->den_law == NF_DEN_AGGLOM) {
    if (p->n_agg < 1 || !(p->agg_sigma > 0.0) || !(p->agg_peak >= 1.0))
      return fail(nullptr, NF_E_INVALID, "agglomerates need n_agg >= 1, sigma > 0, peak >= 1");
  } else if (p->den_law == NF_DEN_MESH) {
    if (!p->den_mesh) return fail(nullptr, NF_E_INVALID, "the mesh density law needs den_mesh");
    uint64_t nv = 1;
    for (int d = 0; d < 3; ++d) {
      if (p->den_ext[d] < 1 || p->den_ext[d] > 4096)
        return fail(nullptr, NF_E_INVALID, "density map extents must be 1..4096");
      nv *= (uint64_t)p->den_ext[d];
    }
    double sum = 0.0;
    for (uint64_t i = 0; i < nv; ++i) {
      const float v = p->den_mesh[i];
      if (!(v >= 0.0f && v <= 1.0f))
        return fail(nullptr, NF_E_INVALID, "density map values must lie in [0, 1]");
      sum += v;
    }
    if (!(sum > 0.0)) return fail(nullptr, NF_E_INVALID, "density map is zero everywhere");
  } else if (p->den_law != NF_DEN_UNIFORM) {
    return fail(nullptr, NF_E_INVALID, "unknown density law");
  }
  if (!(p->soft_frac > 0.0) || p->sep < 0.0) return fail(nullptr, NF_E_INVALID, "bad hard core");
  {
    // periodic images per axis stay bounded: rod reach at most 16 box edges
    const double lmax = p->len_law == NF_LEN_LOGNORMAL ? p->len_max : p->len;
    const double reach = lmax + 2.0 * p->radius * p->soft_frac + p->sep + p->contact_gap;
    const double bmin = std::min(p->box[0], std::min(p->box[1], p->box[2]));
    if (reach > 16.0 * bmin) return fail(nullptr, NF_E_INVALID, "rods longer than 16 box edges");
  }
  const double V = p->box[0] * p->box[1] * p->box[2];
  const double PI = 3.14159265358979323846;
  if (p->n_rods == 0) {
    // simPrms::set_numCNT (src/simPrms.cpp:987-1002): N = ceil(vf V / (pi a^2 l))
    const double vcnt = PI * p->radius * p->radius * p->len;
    const double n = std::ceil(p->vol_frac * V / vcnt);
    if (!(n >= 1.0) || n > 4.0e9) return fail(nullptr, NF_E_INVALID, "rod count out of range");
    p->n_rods = (uint32_t)n;
  }
  if (p->min_batch == 0) p->min_batch = 64;
  if (p->max_batch == 0) {
    const double vex = excluded_volume(p->len, p->radius);
    // three excluded volumes' worth of candidates per round: on average a
    // candidate's excluded volume holds three others of its round.  Fewer,
    // larger rounds cost less than the extra same-round rejections
    // (measured on MI355X: 500k-rod packing 4.77 -> 4.17 ms, 5 -> 3 rounds;
    // 8M-rod packing 103 -> 91 ms, 19 -> 9 rounds; the 256-packing batch
    // 281 -> 290 ms)
    double m = 3.0 * V / vex;
    const double cap = 4.0 * (double)p->n_rods + 1024.0;
    if (m > cap) m = cap;
    if (m > (double)(1u << 23)) m = (double)(1u << 23);
    if (m < 256.0) m = 256.0;
    p->max_batch = (uint32_t)m;
  }
  if (p->min_batch > p->max_batch) p->min_batch = p->max_batch;
  if (p->max_rounds == 0) p->max_rounds = 1000;
  if (p->stall_rounds == 0) p->stall_rounds = 8;
  if (p->precision != NF_PREC_FP64 && p->precision != NF_PREC_FP32_RECHECK)
    return fail(nullptr, NF_E_INVALID, "unknown precision");
  if (p->elec_axis < 0 || p->elec_axis > 2) return fail(nullptr, NF_E_INVALID, "elec_axis must be 0..2");
  return NF_OK;
}

// ===========================================================================
// stencils
// ===========================================================================
namespace nf {
std::vector<int4> build_stencil(const int32_t nc[3], const double box[3], double reach, bool half, int bx) {
  std::vector<std::pair<float, int4>> v;
  const double rm = reach + (double)CELL_MARGIN;
  if (bx < 1 || (half && bx != 1)) bx = 1;
  int k[3];
  double E[3];
  for (int d = 0; d < 3; ++d) {
    E[d] = box[d] / nc[d];
    k[d] = (int)std::floor(rm / E[d]) + 1;
  }
  for (int dz = -k[2]; dz <= k[2]; ++dz)
    for (int dy = -k[1]; dy <= k[1]; ++dy)
      for (int dx = -k[0]; dx <= k[0] + bx - 1; ++dx) {
        if (half) {
          const bool pos = dz > 0 || (dz == 0 && (dy > 0 || (dy == 0 && dx >= 0)));
          if (!pos) continue;
        }
        // whole cells between the offset cell and the block, per axis
        const int gap[3] = {dx >= bx ? dx - bx : (dx < 0 ? -dx - 1 : 0), std::abs(dy) - 1, std::abs(dz) - 1};
        double m2 = 0.0;
        for (int d = 0; d < 3; ++d) {
          const int a = gap[d];
          if (a > 0) m2 += (a * E[d]) * (a * E[d]);
        }
        if (m2 <= rm * rm) {
          // store a slightly low minimum distance so float rounding never prunes
          const float md2 = (float)(m2 * (1.0 - 1e-6));
          int4 e;
          e.x = dx;
          e.y = dy;
          e.z = dz;
          e.w = 0;
          std::memcpy(&e.w, &md2, sizeof(float));
          v.push_back({md2, e});
        }
      }
  std::stable_sort(v.begin(), v.end(), [](const std::pair<float, int4>& a, const std::pair<float, int4>& b) {
    return a.first < b.first;
  });
  std::vector<int4> out;
  out.reserve(v.size());
  for (auto& e : v) out.push_back(e.second);
  return out;
}
}  // namespace nf

// ===========================================================================
// lifecycle
// ===========================================================================
// Crossing lists of an instance (nf_walk.hip).  Fine cells of 1.5 times the
// mean spacing of the rods, between a sixteenth and two thirds of a typical
// rod: 1, 1.5 and 2 times gave 54.7, 52.7 and 56.4 ms of kernels for 32 uneven
// packings, 2.03, 1.89 and 1.91 ms for 500,000 rods (smaller cells: fewer
// pairs, more entries to make).
//
// Which packings: entering a rod costs some seven device-scope atomics, the
// cell-pair engine a number of staged pairs that grows with crowding (rods
// per excluded volume), with the spread of the lengths (its cells are as wide
// as the longest), with the rounds and, where every pair that the filter leaves
// is evaluated in FP64, with the precision.  Rods of one length take the lists
// from this many per excluded volume on; whole generations, cells of one reach
// against lists, at 0.31 / 0.52 / 0.83 / 1.25 / 1.66 / 2.1 / 2.7 in ms:
//   FP32   100,000  .30 .61 .82 1.08 1.40 1.87 2.85    .32 .51 .74  .90 1.14 1.59 2.28
//          300,000  .41 .82 1.27 1.50 2.06 2.64 4.07   .46 .80 1.11 1.36 1.77 2.26 3.10
//          450,000  .45 .93 1.50 1.76 2.44 3.26 5.28   .59 1.01 1.40 1.71 2.22 2.71 3.96
//          1M       .77 1.33 2.14 2.75 4.09 5.69 9.49  1.10 1.83 2.47 3.14 4.25 5.34 7.21
//          4M       2.43 3.84 5.83 8.50 12.9 20.0 31.1 4.14 6.60 8.68 11.6 15.1 19.0 24.5
//          8M       6.63 7.55 9.93 15.7 21.5 32.8 59.2 10.2 12.0 16.1 21.2 27.3 33.9 48.6
//   FP64   700,000  .83 1.81 2.96 3.40 4.87 6.26 9.86  .82 1.34 1.84 2.31 3.08 3.78 5.18
//          1M       .97 2.02 3.25 3.86 5.67 7.49 12.0  1.09 1.81 2.46 3.09 4.18 5.31 7.12
//          1.5M     1.27 2.39 3.82 4.82 7.13 9.63 15.5 1.60 2.58 3.46 4.36 5.86 7.49 9.79
//          2.5M     1.80 3.17 5.11 6.86 10.1 14.2 21.8 2.77 4.21 5.71 7.34 9.87 12.2 15.8
//          4M       2.60 4.45 6.88 9.71 14.4 21.3 32.8 4.13 6.53 8.65 11.5 14.8 19.0 24.3
//          8M       6.97 7.73 10.7 16.6 22.5 33.6 59.0 9.69 11.7 15.8 21.1 27.0 33.8 47.7
// Dense places cost the cells more and take more rounds, so above 300,000 rods
// the line falls with the densest place over the mean: of 16 agglomerates, FP32,
// peak 3 (2.8 over the mean) 4M rods at 1.66 / 2.0 11.8 / 16.7 against 12.8 /
// 16.0 ms, 8M at 2.0 32.8 against 31.8; peak 8 (6.6) 1M at 0.9 / 1.3 3.8 / 5.6
// against 3.5 / 4.8, 4M at 0.9 / 1.3 / 1.7 11.1 / 14.9 / 20.8 against 11.8 / 14.0
// / 18.5; FP64, 4M, peak 3 at 1.3 / 1.66 9.9 / 13.6 against 10.2 / 12.7, peak 8
// at 0.9 13.2 against 11.5.  At peak 20 (16) the lists, as long everywhere as in
// the densest place, take 2.5 GB at 4M rods and lose again: 29 against 41 ms at
// 1.3, where 1M rods still take 11.0 against 7.9.
// Log-normal lengths take them always: at 0.3 / 1 / 2.1 100,000 rods .42 1.37 2.59
// against .32 .85 1.32 ms, 4M 7.2 21.1 54.7 against 4.4 10.9 19.0.
static double lists_from(uint32_t n, bool fp64, double dense) {
  double c = 0.0;
  if (fp64)
    c = n <= 700000u ? 0.0 : n <= 1000000u ? 0.4 : n <= 2000000u ? 0.65 : n <= 3000000u ? 1.55 : 1.9;
  else
    c = n <= 100000u ? 0.0 : n <= 300000u ? 0.4 : n <= 500000u ? 0.75 : n <= 1000000u ? 1.65 : 2.05;
  if (n <= 300000u || (n > 1000000u && dense > 10.0)) return c;
  return c / (1.0 + 0.1 * (std::min(dense, 10.0) - 1.0));
}

// An instance's crossing lists.  peak: densest point over the background or the
// mean, a bound that cell capacities follow; d.dense has it over the mean.
static void plan_fine(const nf_params& p, InstDesc& d, double peak) {
  FineGrid& g = d.fine;
  const double V = p.box[0] * p.box[1] * p.box[2];
  const double crowd = (double)p.n_rods * excluded_volume(p.len, p.radius) / V;
  if (p.len_law == NF_LEN_CONST && crowd < lists_from(p.n_rods, p.precision == NF_PREC_FP64, d.dense)) return;
  const double r = 0.50001 * (double)d.R_max + 16.0 * (double)d.ew;
  double E = 1.5 * std::cbrt(V / (double)p.n_rods);
  E = std::min(std::max(E, p.len / 16.0), p.len / 1.5);
  E = std::max(E, 4.0 * r);
  uint64_t cells = 1;
  for (int a = 0; a < 3; ++a) {
    // one wrap per axis; a grid that uses the whole box
    if (!((double)d.hl_max * 1.0001 + r < 0.999 * p.box[a])) return;
    const double n = std::min(std::max(std::floor(p.box[a] / E), 1.0), 1024.0);
    g.n[a] = (int32_t)n;
    g.e[a] = (float)(p.box[a] / n);
    g.ie[a] = (float)(n / p.box[a]);
    cells *= (uint64_t)g.n[a];
  }
  if (cells > (1ull << ENTRY_BITS) || p.max_batch > (1u << ENTRY_BITS)) return;
  g.r = (float)r;
  // rods crossing a cell: a rod of length l crosses about 2 (3/4 l / E + 1)
  const double lam = peak * (double)p.n_rods / (double)cells * 2.0 * (0.75 * p.len / E + 1.0);
  const double first = std::min((double)p.max_batch, 1.25 * (double)p.n_rods) / (double)p.n_rods;
  auto room = [](double l) { return (uint32_t)std::min(4.0 * std::ceil((1.15 * l + 6.0 * std::sqrt(l) + 10.0) / 4.0), 65532.0); };
  g.capA = room(lam);
  g.capP = room(lam * first);
  g.on = 1u;
}

static int plan_instance(const nf_params& p, InstDesc& d, std::vector<double>& agg,
                         std::vector<int4>& stencil) {
  std::memset(&d, 0, sizeof(d));
  SampleDesc& s = d.smp;
  for (int a = 0; a < 3; ++a) s.box[a] = p.box[a];
  s.len = p.len;
  s.len_sigma = p.len_sigma;
  s.len_min = p.len_min;
  s.len_max = p.len_max;
  s.radius = p.radius;
  s.sep = p.sep;
  s.soft_frac = p.soft_frac;
  s.kappa = p.kappa;
  for (int a = 0; a < 3; ++a) s.axis[a] = p.axis[a];
  if (p.ort_law == NF_ORT_VMF) vmf_basis(s.axis, s.e1, s.e2);
  s.agg_sigma = p.agg_sigma;
  s.agg_peak = p.agg_peak;
  s.seed = p.seed;
  s.stream = p.stream;
  s.len_law = p.len_law;
  s.ort_law = p.ort_law;
  s.den_law = p.den_law;
  s.n_agg = p.den_law == NF_DEN_AGGLOM ? p.n_agg : 0;
  s.agg = nullptr;
  s.mesh = nullptr;  // device copy, set at upload
  for (int a = 0; a < 3; ++a) s.mext[a] = p.den_law == NF_DEN_MESH ? p.den_ext[a] : 0;
  agg.resize(3 * (size_t)s.n_agg);
  for (int k = 0; k < s.n_agg; ++k) agg_centre(p.seed, p.stream, p.box, (uint32_t)k, &agg[3 * k]);

  const float lmaxf = (float)(p.len_law == NF_LEN_LOGNORMAL ? p.len_max : p.len);
  const float af = (float)p.radius;
  d.hl_max = 0.5f * lmaxf;
  const double Rmax = p.soft_frac * ((double)af + (double)af) + p.sep;
  d.R_max = (float)Rmax * 1.000001f;
  const double reach = ((double)d.hl_max + (double)d.hl_max) * REACH_PAD + Rmax;
  // cell edge: requested, or about one typical reach; when that would put
  // more than 256 rods in an average cell (long rods, small boxes) the edge
  // drops towards ~32 rods per cell, but not below a quarter of the reach
  // (a negative cell_size scales that default edge)
  double target = p.cell_size;
  const double V = p.box[0] * p.box[1] * p.box[2];
  if (!(target > 0.0)) {
    // 0.85 of a typical reach: the reject-vs-accepted pass stages the rods
    // of every cell within reach of the home cell, so slightly smaller cells
    // stage fewer far rods (measured optimum on the 500k-rod workload)
    const double e = default_cell_edge(p.len * REACH_PAD + Rmax, (double)p.n_rods / V, 0.85);
    target = target < 0.0 ? -target * e : e;
  }
  double peak = p.den_law == NF_DEN_AGGLOM ? p.agg_peak : 1.0;
  if (p.den_law == NF_DEN_MESH) {
    // densest point relative to the mean of the map
    const uint64_t nv = (uint64_t)p.den_ext[0] * p.den_ext[1] * p.den_ext[2];
    double sum = 0.0, mx = 0.0;
    for (uint64_t i = 0; i < nv; ++i) {
      sum += p.den_mesh[i];
      mx = std::max(mx, (double)p.den_mesh[i]);
    }
    peak = mx * (double)nv / sum;
  }
  const double Lmax = std::max(p.box[0], std::max(p.box[1], p.box[2]));
  d.ew = (float)(5.9604644775390625e-8 * (Lmax + reach) * 1.01);
  double dense = peak;
  if (p.den_law == NF_DEN_AGGLOM) {  // the mean, as if no two agglomerates overlapped
    const double blobs = p.n_agg * std::pow(2.0 * M_PI, 1.5) * p.agg_sigma * p.agg_sigma * p.agg_sigma / V;
    dense /= 1.0 + (peak - 1.0) * std::min(blobs, 1.0);
  }
  d.dense = (float)dense;
  plan_fine(p, d, peak);
  auto cells_of = [&](double edge, int32_t nc[3]) {
    uint64_t c = 1;
    for (int a = 0; a < 3; ++a) {
      nc[a] = (int32_t)std::min(std::max(std::floor(p.box[a] / edge), 1.0), 1024.0);
      c *= (uint64_t)nc[a];
    }
    return c;
  };
  uint64_t ncells = cells_of(target, d.grid);
  if (ncells > (1ull << 26)) return NF_E_INVALID;
  for (int a = 0; a < 3; ++a) d.ncell[a] = d.grid[a];
  // The passes' own grid.  Rods of one length that stay with the cell-pair
  // engine, no cell size asked for: cells just over one reach, whose stencil is
  // the 27 cells around (0.85 of a reach: 81 of 125).  Generation of 1M and 4M
  // rods at half a rod per excluded volume 2.36 -> 1.77 and 7.3 -> 4.7 ms.
  if (!d.fine.on && p.len_law == NF_LEN_CONST && p.cell_size == 0.0)
    ncells = cells_of(default_cell_edge(reach + 2.0 * (double)CELL_MARGIN, (double)p.n_rods / V, 1.0), d.ncell);
  for (int a = 0; a < 3; ++a) {
    d.boxf[a] = (float)p.box[a];
    d.cell_scale[a] = (double)d.ncell[a] / p.box[a];
    d.edge[a] = (float)(p.box[a] / d.ncell[a]);
  }
  d.ncells = (uint32_t)ncells;
  // full stencil, then the half stencil of the same-round pass
  stencil = build_stencil(d.ncell, p.box, reach, false);
  d.st_n = (uint32_t)stencil.size();
  const std::vector<int4> half = build_stencil(d.ncell, p.box, reach, true);
  d.hst_n = (uint32_t)half.size();
  stencil.insert(stencil.end(), half.begin(), half.end());
  // per-cell capacity for accepted rods
  const double cellV = V / (double)ncells;
  const double lam = (double)p.n_rods * cellV / V * peak;
  double cap = std::ceil(lam * 1.25 + 8.0 * std::sqrt(lam) + 16.0);
  if (cap > (double)p.n_rods + 16.0) cap = (double)p.n_rods + 16.0;
  d.cap = (uint32_t)cap;
  d.n_target = p.n_rods;
  d.min_batch = p.min_batch;
  d.max_batch = p.max_batch;
  d.max_rounds = p.max_rounds;
  d.stall_rounds = p.stall_rounds;
  d.sf64 = p.soft_frac;
  d.sep64 = p.sep;
  d.sf32 = (float)p.soft_frac;
  d.sep32 = (float)p.sep;
  return NF_OK;
}

static void release_gen(nf_handle* h) {
  GenBuffers& b = h->gb;
  void* ptrs[] = {b.desc, b.st, b.ri, b.slot_base, b.stencil, b.agg, b.mesh, b.cell_inst, b.oP, b.oD,
                  b.oid, b.ostart, b.ocount, b.ohl, b.bP, b.bD, b.sP, b.sD, b.scell, b.srk,
                  b.surv, b.srank, b.pP, b.pD, b.pslot, b.palive, b.pcount, b.pstart, b.phl,
                  b.items, b.qcnt, b.aP, b.aD, b.aslot, b.aidx, b.acount, b.astart, b.queues, b.scan_tmp,
                  b.fcountA, b.fcountP, b.flistA, b.flistP, b.sdst, b.oR, b.aR};
  for (void* p : ptrs) dfree(h, p);
  b = GenBuffers();
}

void nf::release_contacts(nf_handle* h) {
  ContactBuffers& c = h->cb;
  void* ptrs[] = {c.cP, c.cD, c.cid, c.cstart, c.ccount, c.chl, c.cmask, c.stencil, c.cnt,
                  c.rowptr, c.I, c.J, c.gap, c.gap64, c.img, c.area, c.labels, c.nrow, c.ncol, c.nval,
                  c.nd_pflag, c.nd_edge_a, c.nd_edge_b, c.nd_esrc, c.nd_esnk, c.nd_src_node,
                  c.nd_snk_node, c.nd_egs, c.nd_egk, c.nd_node_rod, c.nd_node_t, c.nd_seg_a,
                  c.nd_seg_b, c.nd_seg_L, c.nd_seg_A, c.nd_ce_a, c.nd_ce_b, c.nd_ce_k, c.nd_cel_node,
                  c.nd_cel_gap, c.nd_cel_side};
  for (void* p : ptrs) dfree(h, p);
  c = ContactBuffers();
}

// Offsets and device memory of the crossing lists of the instances that have
// them (desc: to be uploaded afterwards).
constexpr uint32_t LIST_CAP_MAX = 8192;
constexpr uint64_t LIST_ENTRIES_MAX = (uint64_t)1 << 32;  // 16 GiB
static void free_lists(nf_handle* h) {
  GenBuffers& b = h->gb;
  void* old[] = {b.fcountA, b.fcountP, b.flistA, b.flistP, b.oR, b.aR};
  for (void* p : old) dfree(h, p);
  b.fcountA = b.fcountP = b.flistA = b.flistP = nullptr;
  b.oR = b.aR = nullptr;
  b.total_fine = b.total_listA = b.total_listP = 0;
  b.walk = b.cellwise = false;
}

static int layout_lists(nf_handle* h) {
  GenBuffers& b = h->gb;
  free_lists(h);
  bool walk = false;
  for (InstDesc& d : h->desc) {
    FineGrid& g = d.fine;
    if (!g.on) {
      b.cellwise = true;
      continue;
    }
    const uint64_t cells = (uint64_t)g.n[0] * g.n[1] * g.n[2];
    // entries name a cell slot of the instance in ENTRY_BITS bits; lists far
    // longer than planned (one crowded spot) or past the memory set aside go
    // without
    if ((uint64_t)d.ncells * d.cap > (1ull << ENTRY_BITS) || g.capA > LIST_CAP_MAX || g.capP > LIST_CAP_MAX ||
        b.total_listA + b.total_listP + cells * ((uint64_t)g.capA + g.capP) > LIST_ENTRIES_MAX ||
        b.total_fine + cells > 0xFFFFFFF0ull) {
      g.on = 0u;
      b.cellwise = true;
      continue;
    }
    g.base = (uint32_t)b.total_fine;
    g.offA = b.total_listA;
    g.offP = b.total_listP;
    b.total_fine += cells;
    b.total_listA += cells * g.capA;
    b.total_listP += cells * g.capP;
    walk = true;
  }
  if (!walk) return NF_OK;
  int rc = dalloc(h, &b.fcountA, b.total_fine);
  if (rc == NF_OK) rc = dalloc(h, &b.fcountP, b.total_fine);
  if (rc == NF_OK) rc = dalloc(h, &b.flistA, b.total_listA);
  if (rc == NF_OK) rc = dalloc(h, &b.flistP, b.total_listP);
  if (rc == NF_OK) rc = dalloc(h, &b.oR, 2 * b.total_old);
  if (rc == NF_OK) rc = dalloc(h, &b.aR, 2 * b.T_cap);
  if (rc == NF_E_NOMEM) {
    // the packings do not need the lists
    for (InstDesc& d : h->desc) d.fine.on = 0u;
    return layout_lists(h);
  }
  b.walk = rc == NF_OK;  // (not before: shed_lists)
  return rc;
}

static void drop_graph(nf_handle* h);

// Memory has run out: the lists give theirs to the call that needs it, and the
// generations that follow go without (a third of a large handle's memory, up to
// 16 GiB).  False if there are none, or a pass is using them.
static bool nf::shed_lists(nf_handle* h) {
  GenBuffers& b = h->gb;
  if (!b.walk || h->lists_in_use) return false;
  for (InstDesc& d : h->desc) d.fine.on = 0u;
  free_lists(h);
  b.cellwise = true;
  drop_graph(h);
  trace("out of memory: crossing lists given back");
  return hipMemcpy(b.desc, h->desc.data(), sizeof(InstDesc) * h->desc.size(), hipMemcpyHostToDevice) == hipSuccess;
}

extern "C" int nf_create_batch(const nf_params* ps, int n, nf_handle** out) {
  if (!out) return fail(nullptr, NF_E_INVALID, "null output handle");
  *out = nullptr;
  if (!ps || n < 1 || n > 65536) return fail(nullptr, NF_E_INVALID, "need 1..65536 instances");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1)
    return fail(nullptr, NF_E_NODEVICE, "no HIP device visible");
  nf_handle* h = new nf_handle();
  h->params.assign(ps, ps + n);
  for (int i = 0; i < n; ++i) {
    int rc = nf_params_normalize(&h->params[i]);
    if (rc != NF_OK) {
      std::string m = "instance " + std::to_string(i) + ": " + g_last_error;
      delete h;
      return fail(nullptr, rc, m);
    }
  }
  (void)hipGetDevice(&h->device);
  if (hipStreamCreateWithFlags(&h->stream, hipStreamNonBlocking) != hipSuccess) {
    delete h;
    return fail(nullptr, NF_E_HIP, "hipStreamCreate failed");
  }
  for (auto& e : h->ev) (void)hipEventCreate(&e);

  // plan all instances
  h->desc.resize(n);
  std::vector<std::vector<double>> aggs(n);
  std::vector<std::vector<int4>> sts(n);
  GenBuffers& b = h->gb;
  b.n_inst = n;
  uint64_t cell_base = 0, old_off = 0, rod_off = 0, T_cap = 0, agg_total = 0, st_total = 0,
           mesh_total = 0;
  for (int i = 0; i < n; ++i) {
    InstDesc& d = h->desc[i];
    if (plan_instance(h->params[i], d, aggs[i], sts[i]) != NF_OK) {
      delete h;
      return fail(nullptr, NF_E_INVALID, "instance " + std::to_string(i) + ": cell grid too large");
    }
    d.cell_base = (uint32_t)cell_base;
    d.old_off = old_off;
    d.rod_off = (uint32_t)rod_off;
    d.st_off = (uint32_t)st_total;
    d.hst_off = (uint32_t)st_total + d.st_n;
    cell_base += d.ncells;
    old_off += (uint64_t)d.ncells * d.cap;
    rod_off += d.n_target;
    T_cap += d.max_batch;
    agg_total += aggs[i].size();
    if (h->params[i].den_law == NF_DEN_MESH)
      mesh_total += (uint64_t)d.smp.mext[0] * d.smp.mext[1] * d.smp.mext[2];
    st_total += sts[i].size();
    if (cell_base > 0xFFFFFFF0ull || old_off > 0xFFFFFFF0ull || rod_off > 0xFFFFFFF0ull ||
        T_cap > 0xFFFFFFF0ull) {
      delete h;
      return fail(nullptr, NF_E_INVALID, "batch exceeds 32-bit index space");
    }
  }
  b.total_cells = cell_base;
  b.total_old = old_off;
  b.total_rods = rod_off;
  b.T_cap = T_cap;
  int rc = NF_OK;
#define ALLOC(p, n_)                      \
  if (rc == NF_OK) rc = dalloc(h, &(p), (n_));
  ALLOC(b.desc, n);
  ALLOC(b.st, n);
  ALLOC(b.ri, 1);
  ALLOC(b.slot_base, n + 1);
  ALLOC(b.stencil, st_total);
  ALLOC(b.agg, agg_total);
  ALLOC(b.mesh, mesh_total);
  ALLOC(b.cell_inst, b.total_cells);
  ALLOC(b.oP, b.total_old);
  ALLOC(b.oD, b.total_old);
  ALLOC(b.oid, b.total_old);
  ALLOC(b.ostart, b.total_cells);
  ALLOC(b.ocount, b.total_cells);
  ALLOC(b.ohl, b.total_cells);
  ALLOC(b.bP, b.total_rods);
  ALLOC(b.bD, b.total_rods);
  ALLOC(b.sP, b.T_cap);
  ALLOC(b.sD, b.T_cap);
  ALLOC(b.scell, b.T_cap);
  ALLOC(b.srk, b.T_cap);
  ALLOC(b.surv, b.T_cap + 1);
  ALLOC(b.srank, b.T_cap + 1);
  ALLOC(b.pP, b.T_cap);
  ALLOC(b.pD, b.T_cap);
  ALLOC(b.pslot, b.T_cap);
  ALLOC(b.palive, b.T_cap);
  ALLOC(b.pcount, b.total_cells);
  ALLOC(b.pstart, b.total_cells + 1);
  ALLOC(b.items, b.total_cells * pair_items_max(b.total_cells));
  ALLOC(b.qcnt, QUEUES_PER_KERNEL);
  ALLOC(b.aP, b.T_cap);
  ALLOC(b.aD, b.T_cap);
  ALLOC(b.aslot, b.T_cap);
  ALLOC(b.aidx, b.T_cap + 1);
  ALLOC(b.acount, b.total_cells);
  ALLOC(b.astart, b.total_cells + 1);
  ALLOC(b.phl, b.total_cells);
  ALLOC(b.queues, Q_N * QWORDS);
  ALLOC(b.sdst, b.T_cap);
  ALLOC(b.scan_tmp, std::max(scan_tmp_words(b.total_cells), scan_tmp_words(b.T_cap)));
#undef ALLOC
  if (rc == NF_OK) rc = layout_lists(h);
  if (rc != NF_OK) {
    std::string m = h->err;
    nf_destroy(h);
    return fail(nullptr, rc, m);
  }
  // upload descriptors, agglomerates, stencils, per-cell tables
  std::vector<double> agg_all;
  std::vector<float> mesh_all;
  std::vector<int4> st_all;
  std::vector<uint32_t> cinst(b.total_cells), ostart(b.total_cells);
  for (int i = 0; i < n; ++i) {
    InstDesc& d = h->desc[i];
    d.smp.agg = aggs[i].empty() ? nullptr : b.agg + agg_all.size();
    agg_all.insert(agg_all.end(), aggs[i].begin(), aggs[i].end());
    if (h->params[i].den_law == NF_DEN_MESH) {
      const uint64_t nv = (uint64_t)d.smp.mext[0] * d.smp.mext[1] * d.smp.mext[2];
      d.smp.mesh = b.mesh + mesh_all.size();
      mesh_all.insert(mesh_all.end(), h->params[i].den_mesh, h->params[i].den_mesh + nv);
      h->params[i].den_mesh = nullptr;  // the caller's buffer: not kept past nf_create
    }
    st_all.insert(st_all.end(), sts[i].begin(), sts[i].end());
    for (uint32_t c = 0; c < d.ncells; ++c) {
      cinst[d.cell_base + c] = (uint32_t)i;
      ostart[d.cell_base + c] = (uint32_t)(d.old_off + (uint64_t)c * d.cap);
    }
  }
  hipError_t e = hipSuccess;
  if (e == hipSuccess) e = hipMemcpy(b.desc, h->desc.data(), sizeof(InstDesc) * n, hipMemcpyHostToDevice);
  if (e == hipSuccess && !agg_all.empty())
    e = hipMemcpy(b.agg, agg_all.data(), sizeof(double) * agg_all.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess && !mesh_all.empty())
    e = hipMemcpy(b.mesh, mesh_all.data(), sizeof(float) * mesh_all.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess && !st_all.empty())
    e = hipMemcpy(b.stencil, st_all.data(), sizeof(int4) * st_all.size(), hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b.cell_inst, cinst.data(), sizeof(uint32_t) * b.total_cells, hipMemcpyHostToDevice);
  if (e == hipSuccess)
    e = hipMemcpy(b.ostart, ostart.data(), sizeof(uint32_t) * b.total_cells, hipMemcpyHostToDevice);
  if (e != hipSuccess) {
    nf_destroy(h);
    return fail(nullptr, NF_E_HIP, std::string("upload failed: ") + hipGetErrorString(e));
  }
  h->n_rods.assign(n, 0);
  h->given.assign(n, RodMean{0.0, 0.0});
  h->short_gap.assign(n, HUGE_VAL);
  h->planned_cap.resize(n);
  h->planned_list.resize(n);
  for (int i = 0; i < n; ++i) {
    h->planned_cap[i] = h->desc[i].cap;
    h->planned_list[i] = {h->desc[i].fine.capA, h->desc[i].fine.capP};
  }
  *out = h;
  return NF_OK;
}

extern "C" int nf_create(const nf_params* p, nf_handle** out) { return nf_create_batch(p, 1, out); }

extern "C" void nf_destroy(nf_handle* h) {
  if (!h) return;
  if (h->stream) (void)hipStreamSynchronize(h->stream);
  if (h->graph) (void)hipGraphExecDestroy(h->graph);
  release_contacts(h);
  release_gen(h);
  trim_pool(h);
  for (auto& kv : h->allocs)
    if (!slab_of(h, kv.first)) (void)hipFree(kv.first);
  for (auto& slabs : h->slabs)
    for (auto& s : slabs) (void)hipFree(s.p);
  for (auto& e : h->ev)
    if (e) (void)hipEventDestroy(e);
  release_pinned(h);
  if (h->stream) (void)hipStreamDestroy(h->stream);
  delete h;
}

extern "C" const char* nf_last_error(const nf_handle* h) {
  return h ? h->err.c_str() : g_last_error.c_str();
}

extern "C" int nf_num_instances(const nf_handle* h) { return h ? (int)h->params.size() : 0; }

extern "C" const char* nf_version(void) { return "nanofiller-mi355x 0.1 (gfx950)"; }

static int scale_slots(nf_handle* h, double scale);

// A captured round graph holds the launch shapes and buffers of its capture.
static void drop_graph(nf_handle* h) {
  if (h->graph) {
    (void)hipGraphExecDestroy(h->graph);
    h->graph = nullptr;
  }
}

extern "C" int nf_set_option(nf_handle* h, int key, int64_t value) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  switch (key) {
    case NF_OPT_GRAPH: h->opt_graph = value ? 1 : 0; break;
    case NF_OPT_PROFILE: h->opt_profile = value ? 1 : 0; break;
    case NF_OPT_DIAG: h->opt_diag = value ? 1 : 0; break;
    case NF_OPT_CONTACT_PREC:
      if (value != -1 && value != NF_PREC_FP64 && value != NF_PREC_FP32_RECHECK)
        return fail(h, NF_E_INVALID, "bad contact precision");
      h->opt_contact_prec = (int)value;
      break;
    case NF_OPT_CONTACT_ENGINE:
      if (value != NF_ENGINE_FOOTPRINT && value != NF_ENGINE_CELLS)
        return fail(h, NF_E_INVALID, "bad contact engine");
      h->opt_contact_engine = (int)value;
      break;
    case NF_OPT_FOOTPRINT_FINE:
      if (value < 0 || value > 1000000) return fail(h, NF_E_INVALID, "footprint fine cell factor out of range");
      h->opt_footprint_fine = (int)value;
      break;
    case NF_OPT_WAVES_OLD:
    case NF_OPT_WAVES_NEW:
      if (value < 0 || value > 16) return fail(h, NF_E_INVALID, "waves per CU out of range (0..16)");
      (key == NF_OPT_WAVES_OLD ? h->gb.tiles.waves_old : h->gb.tiles.waves_new) = (uint32_t)value;
      drop_graph(h);
      break;
    case NF_OPT_PART_SHIFT:
      if (value < -1 || value > 3) return fail(h, NF_E_INVALID, "part shift out of range (-1..3)");
      h->gb.tiles.part_shift = (int32_t)value;
      drop_graph(h);
      break;
    case NF_OPT_SPLIT_MIN:
      if (value < 0 || value > 4096) return fail(h, NF_E_INVALID, "split minimum out of range (0..4096)");
      h->gb.tiles.split_min = (uint32_t)value;
      drop_graph(h);
      break;
    case NF_OPT_TEST_ALL_PAIRS:
      h->gb.tiles.test_all = value ? 1u : 0u;
      drop_graph(h);
      break;
    case NF_OPT_CROSSING_LISTS:
      h->gb.tiles.lists = value ? 1u : 0u;
      drop_graph(h);
      break;
    case NF_OPT_SLOT_SCALE:
      if (value < 1 || value > 1000000) return fail(h, NF_E_INVALID, "slot scale out of range (1..1000000)");
      return scale_slots(h, (double)value * 1e-3);
    case NF_OPT_POST_INSTANCE:
      if (value < 0 || value >= (int64_t)h->params.size()) return fail(h, NF_E_INVALID, "no such instance");
      if ((int)value != h->post_inst) {
        release_contacts(h);  // contacts, network and cell lists belong to the previous instance
        h->post_inst = (int)value;
      }
      break;
    case NF_OPT_FOOTPRINT_OCC:
      if (value < 0 || value > 200) return fail(h, NF_E_INVALID, "footprint occupancy out of range (0..200)");
      h->opt_footprint_occ = (int)value;
      break;
    default: return fail(h, NF_E_INVALID, "unknown option");
  }
  return NF_OK;
}

// ===========================================================================
// generation
// ===========================================================================
static int reset_generation(nf_handle* h) {
  h->gb.one_length = true;
  for (const nf_params& p : h->params) h->gb.one_length = h->gb.one_length && p.len_law == NF_LEN_CONST;
  launch_reset(h->gb, h->stream);
  HIPCHK(h, hipGetLastError());
  return NF_OK;
}

static int build_graph(nf_handle* h, int prec, int diag) {
  if (h->graph && h->graph_prec == prec && h->graph_diag == diag) return NF_OK;
  if (h->graph) {
    (void)hipGraphExecDestroy(h->graph);
    h->graph = nullptr;
  }
  hipGraph_t g = nullptr;
  HIPCHK(h, hipStreamBeginCapture(h->stream, hipStreamCaptureModeThreadLocal));
  launch_round(h->gb, prec, diag, h->stream, nullptr);
  hipError_t e = hipStreamEndCapture(h->stream, &g);
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("graph capture: ") + hipGetErrorString(e));
  e = hipGraphInstantiate(&h->graph, g, nullptr, nullptr, 0);
  (void)hipGraphDestroy(g);
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("graph instantiate: ") + hipGetErrorString(e));
  h->graph_prec = prec;
  h->graph_diag = diag;
  return NF_OK;
}

// Milestone dumps (VOLUME_PERCENT_LIST, src/cudaMain.cu:136-142): after a
// round, instance 0's volume fraction from its accepted count; when it has
// reached the next listed value, its packing so far (the accepted rods sit
// at the front of its rod buffer, in acceptance order) is saved as a state
// file named by the fraction reached, and every value reached is passed.
// The reference compares the fraction in percent with the list converted
// to fractions (a hundredfold early trigger) and reads past the list's end
// after its last value; here both are percent and the list ends the dumps.
static int milestone_check(nf_handle* h, size_t* next) {
  if (*next >= h->milestones.size()) return NF_OK;
  InstState st0{};
  HIPCHK(h, hipMemcpy(&st0, h->gb.st, sizeof(InstState), hipMemcpyDeviceToHost));
  // out of room: the round's packing may hold rods that overlap (its lists of
  // survivors were cut short), and the generation starts again, dumps included
  if (st0.overflow != 0u) return NF_OK;
  const nf_params& p = h->params[0];
  const double PI = 3.14159265358979323846;
  const double vf = (double)st0.n_acc * PI * p.radius * p.radius * p.len / (p.box[0] * p.box[1] * p.box[2]) * 100.0;
  if (vf < h->milestones[*next]) return NF_OK;
  char name[64];
  std::snprintf(name, sizeof(name), "state_%4.2f.bin", vf);
  const std::string path = h->milestone_dir.empty() ? std::string(name) : h->milestone_dir + "/" + name;
  const uint32_t keep = h->n_rods[0];
  h->n_rods[0] = st0.n_acc;
  const int rc = nf_save_state(h, path.c_str());
  h->n_rods[0] = keep;
  if (rc != NF_OK) return rc;
  trace("generate: milestone %s (%u rods)", path.c_str(), st0.n_acc);
  while (*next < h->milestones.size() && h->milestones[*next] <= vf) ++*next;
  return NF_OK;
}

extern "C" int nf_set_milestones(nf_handle* h, const double* vf_percent, int32_t n, const char* dir) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  if (n < 0 || (n > 0 && !vf_percent)) return fail(h, NF_E_INVALID, "bad milestone list");
  if (n > 0 && h->params.size() != 1) return fail(h, NF_E_INVALID, "milestones need a single-instance handle");
  std::vector<double> v(vf_percent, vf_percent + n);
  for (size_t i = 0; i < v.size(); ++i)
    if (!(v[i] > 0.0) || (i > 0 && !(v[i] > v[i - 1])))
      return fail(h, NF_E_INVALID, "milestones must be positive and ascending");
  h->milestones = v;
  h->milestone_dir = dir ? dir : "";
  return NF_OK;
}

// Per-cell slots of the accepted rods (the "old" set): instance i gets
// caps[i] slots per cell.  Reallocates the slot arrays, rewrites each
// instance's offset and every cell's first slot, and drops a captured round
// graph (its kernel arguments name the old arrays).  The packing does not
// depend on the capacity, only whether it suffices.
static int relayout_old(nf_handle* h, const std::vector<uint32_t>& caps) {
  GenBuffers& b = h->gb;
  const int n = (int)h->desc.size();
  uint64_t off = 0;
  for (int i = 0; i < n; ++i) {
    InstDesc& d = h->desc[i];
    d.cap = caps[i];
    d.old_off = off;
    off += (uint64_t)d.ncells * d.cap;
  }
  if (off > 0xFFFFFFF0ull) return fail(h, NF_E_INVALID, "cell slots exceed the 32-bit index space");
  free_lists(h);  // laid out anew below
  dfree(h, b.oP);
  dfree(h, b.oD);
  dfree(h, b.oid);
  b.oP = b.oD = nullptr;
  b.oid = nullptr;
  int rc = dalloc(h, &b.oP, std::max<uint64_t>(off, 1));
  if (rc == NF_OK) rc = dalloc(h, &b.oD, std::max<uint64_t>(off, 1));
  if (rc == NF_OK) rc = dalloc(h, &b.oid, std::max<uint64_t>(off, 1));
  if (rc != NF_OK) return rc;
  b.total_old = off;
  rc = layout_lists(h);
  if (rc != NF_OK) return rc;
  std::vector<uint32_t> ostart(b.total_cells);
  for (int i = 0; i < n; ++i) {
    const InstDesc& d = h->desc[i];
    for (uint32_t c = 0; c < d.ncells; ++c) ostart[d.cell_base + c] = (uint32_t)(d.old_off + (uint64_t)c * d.cap);
  }
  HIPCHK(h, hipMemcpy(b.desc, h->desc.data(), sizeof(InstDesc) * n, hipMemcpyHostToDevice));
  HIPCHK(h, hipMemcpy(b.ostart, ostart.data(), sizeof(uint32_t) * b.total_cells, hipMemcpyHostToDevice));
  if (h->graph) {
    (void)hipGraphExecDestroy(h->graph);
    h->graph = nullptr;
  }
  return NF_OK;
}

static uint32_t scaled_list(uint32_t cap, double scale) {
  return (uint32_t)(4.0 * std::max(1.0, std::min(std::ceil(cap * scale / 4.0), LIST_CAP_MAX / 4.0)));
}

// The planned slots per cell and list lengths scaled by scale (at least one, at most what
// cannot overflow: the instance's target + 16).
static int scale_slots(nf_handle* h, double scale) {
  std::vector<uint32_t> caps(h->desc.size());
  for (size_t i = 0; i < caps.size(); ++i) {
    const double c = std::ceil((double)h->planned_cap[i] * scale);
    caps[i] = (uint32_t)std::max(1.0, std::min(c, (double)h->desc[i].n_target + 16.0));
    FineGrid& g = h->desc[i].fine;
    if (!g.on) continue;
    g.capA = scaled_list(h->planned_list[i].first, scale);
    g.capP = scaled_list(h->planned_list[i].second, scale);
  }
  return relayout_old(h, caps);
}

static int generate_once(nf_handle* h, nf_gen_stats* stats, std::vector<std::pair<int, uint32_t>>* overflowed);

// Generation with growth: an instance whose cell slots or crossing lists
// overflowed is generated again from the start with twice the room (the
// packing is the same; only its storage was too small), up to the slots that
// cannot overflow.
extern "C" int nf_generate(nf_handle* h, nf_gen_stats* stats) {
  if (!h) return fail(nullptr, NF_E_INVALID, "null handle");
  uint32_t growths = 0;
  for (;;) {
    std::vector<std::pair<int, uint32_t>> over;  // instance, what ran out of room (OVER_*)
    const int rc = generate_once(h, stats, &over);
    if (rc != NF_E_OVERFLOW || over.empty()) {
      if (stats)
        for (int i = 0; i < h->gb.n_inst; ++i) stats[i].slot_growths = growths;
      return rc;
    }
    std::vector<uint32_t> caps(h->desc.size());
    bool grew = false;
    for (size_t i = 0; i < caps.size(); ++i) caps[i] = h->desc[i].cap;
    for (const auto& [i, bits] : over) {
      if (bits & OVER_SLOTS) {
        const uint32_t lim = h->desc[i].n_target + 16u;
        const uint32_t c = (uint32_t)std::min<uint64_t>(2ull * caps[i], lim);
        grew = grew || c > caps[i];
        caps[i] = c;
      }
      // lists double too; past LIST_CAP_MAX the instance goes without them
      FineGrid& g = h->desc[i].fine;
      if (bits & OVER_LISTS_A) g.capA *= 2u;
      if (bits & OVER_LISTS_P) g.capP *= 2u;
      grew = grew || (bits & (OVER_LISTS_A | OVER_LISTS_P)) != 0u;
    }
    if (!grew) return rc;
    const int r2 = relayout_old(h, caps);
    if (r2 != NF_OK) return r2;
    ++growths;
    trace("generate: out of room (%u), regenerating with %u slots per cell (instance %d)", over[0].second,
          caps[over[0].first], over[0].first);
  }
}

static int generate_once(nf_handle* h, nf_gen_stats* stats, std::vector<std::pair<int, uint32_t>>* overflowed) {
  h->err.clear();
  const int prec = h->params[0].precision;
  for (auto& p : h->params)
    if (p.precision != prec) return fail(h, NF_E_INVALID, "all instances of a batch share one precision");
  int rc = reset_generation(h);
  if (rc) return rc;
  const bool use_graph = h->opt_graph && !h->opt_profile;
  trace("generate: %d instance(s), precision %d, graph %d, profile %d", h->gb.n_inst, prec,
        (int)use_graph, h->opt_profile);
  if (use_graph) {
    rc = build_graph(h, prec, h->opt_diag);
    if (rc) return rc;
    trace("generate: graph built");
  }
  double kern[8] = {0};
  RoundInfo ri{};
  RoundInfo* ri_host = &host_scalars(h)->ri;
  uint32_t max_rounds = 0;
  for (auto& p : h->params) max_rounds = std::max(max_rounds, p.max_rounds);
  const auto t0 = std::chrono::steady_clock::now();
  uint32_t launched = 0;
  int batch = 1;
  std::vector<std::array<hipEvent_t, 8>> prof_ev;
  size_t prof_used = 0;
  size_t next_ms = 0;  // next milestone (volume fraction) to dump
  hipError_t e = hipSuccess;
  for (;;) {
    for (int k = 0; k < batch && e == hipSuccess; ++k) {
      if (use_graph) {
        e = hipGraphLaunch(h->graph, h->stream);
      } else {
        hipEvent_t* ev = nullptr;
        if (h->opt_profile) {
          // one event set per round, read back after the final sync
          if (prof_used == prof_ev.size()) {
            prof_ev.emplace_back();
            for (auto& x : prof_ev.back()) (void)hipEventCreate(&x);
          }
          ev = prof_ev[prof_used++].data();
        }
        launch_round(h->gb, prec, h->opt_diag, h->stream, ev);
        e = hipGetLastError();
      }
      ++launched;
    }
    if (e == hipSuccess) e = scalars_to_host(h, ri_host, h->gb.ri, sizeof(RoundInfo));
    if (e == hipSuccess) e = sync_stream(h->stream, "generation round");
    if (e != hipSuccess) break;
    ri = *ri_host;
    trace("generate: %u rounds launched, controller rounds %u, running %u, last T %u", launched,
          ri.rounds, ri.running, ri.T);
    if (!h->milestones.empty()) {
      const int mrc = milestone_check(h, &next_ms);
      if (mrc != NF_OK) return mrc;
    }
    if (ri.running == 0 || launched > max_rounds + 2) break;
    // next batch: the rounds the controller expects to need at the last
    // round's acceptance (at most 8 between host checks); one at a time
    // while a milestone is pending
    batch = (int)std::min<uint32_t>(std::max<uint32_t>(ri.est, 1u), 8u);
    if (next_ms < h->milestones.size()) batch = 1;
  }
  const auto t1 = std::chrono::steady_clock::now();
  if (e == hipSuccess && h->opt_profile) {
    const int cls[7] = {NF_K_CONTROL, NF_K_GEN, NF_K_BIN, NF_K_REJECT_OLD, NF_K_REJECT_NEW,
                        NF_K_COMMIT, NF_K_CONTROL};
    for (size_t r = 0; r < prof_used; ++r)
      for (int c = 0; c < 7; ++c) {
        float ms = 0.0f;
        if (hipEventElapsedTime(&ms, prof_ev[r][c], prof_ev[r][c + 1]) == hipSuccess) kern[cls[c]] += ms;
      }
  }
  for (auto& a : prof_ev)
    for (auto& x : a) (void)hipEventDestroy(x);
  if (e != hipSuccess) return fail(h, NF_E_HIP, std::string("generation: ") + hipGetErrorString(e));
  const double wall = std::chrono::duration<double, std::milli>(t1 - t0).count();
  std::vector<InstState> st(h->gb.n_inst);
  const HostPart st_part = {st.data(), h->gb.st, sizeof(InstState) * st.size()};
  HIPCHK(h, to_host(h, &st_part, 1));
  int status_rc = NF_OK;
  for (int i = 0; i < h->gb.n_inst; ++i) {
    h->n_rods[i] = st[i].n_acc;
    if (st[i].status == NF_STATUS_OVERFLOW) {
      status_rc = NF_E_OVERFLOW;
      overflowed->push_back({i, st[i].overflow});
    }
    if (stats) {
      nf_gen_stats& s = stats[i];
      std::memset(&s, 0, sizeof(s));
      s.n_target = h->desc[i].n_target;
      s.n_accepted = st[i].n_acc;
      s.rounds = st[i].round;
      s.status = (int32_t)st[i].status;
      s.candidates = st[i].candidates;
      s.proposals = st[i].proposals;
      s.pair_tests = st[i].pair_tests;
      s.rechecks = st[i].rechecks;
      s.rejected_old = st[i].rej_old;
      s.rejected_new = st[i].rej_new;
      s.wall_ms = wall;
      for (int k = 0; k < 8; ++k) s.kern_ms[k] = kern[k];
      s.max_abs_d32_d64 = st[i].max_dd;
      s.tile_bytes = st[i].tile_bytes;
      s.tile_bytes_new = st[i].tile_bytes_new;
      s.rounds_launched = launched;
    }
  }
  h->generated = true;
  h->given.assign(h->given.size(), RodMean{0.0, 0.0});
  h->short_gap.assign(h->short_gap.size(), HUGE_VAL);
  h->cb.valid = false;
  h->cb.net_valid = false;
  h->cb.nd_valid = false;
  if (status_rc != NF_OK) return fail(h, status_rc, "a cell exceeded its capacity during generation");
  return NF_OK;
}

extern "C" int nf_get_rods(nf_handle* h, int inst, float* rods, uint32_t cap, uint32_t* n) {
  if (!h || inst < 0 || inst >= (int)h->params.size()) return fail(h, NF_E_INVALID, "bad instance");
  const uint32_t cnt = h->n_rods[inst];
  if (n) *n = cnt;
  if (!rods) return NF_OK;
  if (cap < cnt) return fail(h, NF_E_CAPACITY, "rod buffer too small");
  const uint32_t off = h->desc[inst].rod_off;
  HIPCHK(h, rods_to_host(h, h->gb.bP + off, h->gb.bD + off, cnt, rods));
  return NF_OK;
}

extern "C" int nf_set_rods(nf_handle* h, int inst, const float* rods, uint32_t n) {
  if (!h || inst < 0 || inst >= (int)h->params.size()) return fail(h, NF_E_INVALID, "bad instance");
  if (n > h->desc[inst].n_target) return fail(h, NF_E_CAPACITY, "more rods than the instance target");
  if (n && !rods) return fail(h, NF_E_INVALID, "null rods");
  for (uint32_t i = 0; i < n; ++i) {
    const float* r = rods + 8 * (size_t)i;
    if (!(r[6] > 0.0f) || !(r[7] > 0.0f)) return fail(h, NF_E_INVALID, "rod length and radius must be > 0");
    for (int a = 0; a < 3; ++a)
      if (!(r[a] >= 0.0f && r[a] < (float)h->params[inst].box[a]))
        return fail(h, NF_E_INVALID, "rod centre outside the box");
  }
  const uint32_t off = h->desc[inst].rod_off;
  HIPCHK(h, rods_to_device(h, rods, n, h->gb.bP + off, h->gb.bD + off));
  h->n_rods[inst] = n;
  // (of some thousand rods: sums over all of 200,000 took 40 us)
  RodMean sum = {0.0, 0.0};
  const uint32_t step = n / 1024u + 1u;
  uint32_t seen = 0;
  for (uint32_t i = 0; i < n; i += step, ++seen) {
    sum.len += rods[8 * (size_t)i + 6];
    sum.radius += rods[8 * (size_t)i + 7];
  }
  h->given[inst] = n ? RodMean{sum.len / seen, sum.radius / seen} : RodMean{0.0, 0.0};
  h->short_gap[inst] = HUGE_VAL;
  h->generated = false;
  h->cb.valid = false;
  h->cb.net_valid = false;
  h->cb.nd_valid = false;
  return NF_OK;
}


extern "C" int nf_get_params(nf_handle* h, int inst, nf_params* out) {
  if (!h || !out || inst < 0 || inst >= (int)h->params.size()) return fail(h, NF_E_INVALID, "bad instance");
  *out = h->params[inst];
  return NF_OK;
}

extern "C" int nf_agglomerate_centres(const nf_params* p, double* out, int32_t cap) {
  if (!p) return fail(nullptr, NF_E_INVALID, "null parameters");
  if (p->den_law != NF_DEN_AGGLOM) return 0;
  if (p->n_agg < 0) return fail(nullptr, NF_E_INVALID, "n_agg must be >= 0");
  if (out && cap < p->n_agg) return fail(nullptr, NF_E_CAPACITY, "buffer too small");
  if (out)
    for (int k = 0; k < p->n_agg; ++k) agg_centre(p->seed, p->stream, p->box, (uint32_t)k, &out[3 * k]);
  return p->n_agg;
}

// ===========================================================================
// diagnostics
// ===========================================================================
extern "C" int nf_selftest(int which, const double* in, double* out, uint64_t n) {
  if (which < 0 || which > 6 || (n && (!in || !out))) return fail(nullptr, NF_E_INVALID, "bad selftest args");
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(nullptr, NF_E_NODEVICE, "no HIP device");
  const uint64_t nin = which == 3 ? 2 * n : n;
  double *din = nullptr, *dout = nullptr;
  if (hipMalloc((void**)&din, sizeof(double) * (nin ? nin : 1)) != hipSuccess)
    return fail(nullptr, NF_E_NOMEM, "hipMalloc failed");
  if (hipMalloc((void**)&dout, sizeof(double) * (n ? n : 1)) != hipSuccess) {
    (void)hipFree(din);
    return fail(nullptr, NF_E_NOMEM, "hipMalloc failed");
  }
  hipError_t e = hipMemcpy(din, in, sizeof(double) * nin, hipMemcpyHostToDevice);
  if (e == hipSuccess && n) {
    launch_selftest(which, din, dout, n, nullptr);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(out, dout, sizeof(double) * n, hipMemcpyDeviceToHost);
  (void)hipFree(din);
  (void)hipFree(dout);
  if (e != hipSuccess) return fail(nullptr, NF_E_HIP, std::string("selftest: ") + hipGetErrorString(e));
  return NF_OK;
}

extern "C" int nf_selftest_pairs(const float* ra, const float* rb, const double* shift, uint64_t n, int contact,
                                 double sep_or_gap, double soft_frac, float ew, int32_t* screen, int32_t* decided,
                                 int32_t* within) {
  if (n && (!ra || !rb || !shift || !screen || !decided || !within))
    return fail(nullptr, NF_E_INVALID, "bad selftest_pairs args");
  if (n == 0) return NF_OK;
  int ndev = 0;
  if (hipGetDeviceCount(&ndev) != hipSuccess || ndev < 1) return fail(nullptr, NF_E_NODEVICE, "no HIP device");
  const size_t fb = sizeof(float) * 8 * n, db = sizeof(double) * 3 * n, ib = sizeof(int32_t) * n;
  char* buf = nullptr;
  if (hipMalloc((void**)&buf, 2 * fb + db + 3 * ib) != hipSuccess) return fail(nullptr, NF_E_NOMEM, "hipMalloc failed");
  float* da = (float*)buf;
  float* dbr = (float*)(buf + fb);
  double* dsh = (double*)(buf + 2 * fb);
  int32_t* o = (int32_t*)(buf + 2 * fb + db);
  hipError_t e = hipMemcpy(da, ra, fb, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dbr, rb, fb, hipMemcpyHostToDevice);
  if (e == hipSuccess) e = hipMemcpy(dsh, shift, db, hipMemcpyHostToDevice);
  if (e == hipSuccess) {
    launch_selftest_pairs(da, dbr, dsh, n, contact, sep_or_gap, soft_frac, ew, o, o + n, o + 2 * n, nullptr);
    e = hipGetLastError();
  }
  if (e == hipSuccess) e = hipDeviceSynchronize();
  if (e == hipSuccess) e = hipMemcpy(screen, o, ib, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(decided, o + n, ib, hipMemcpyDeviceToHost);
  if (e == hipSuccess) e = hipMemcpy(within, o + 2 * n, ib, hipMemcpyDeviceToHost);
  (void)hipFree(buf);
  if (e != hipSuccess) return fail(nullptr, NF_E_HIP, std::string("selftest_pairs: ") + hipGetErrorString(e));
  return NF_OK;
}
