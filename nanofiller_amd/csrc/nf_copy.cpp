// nf_copy.cpp - results to the caller's memory and rods from it, through
// pinned memory that the handle keeps.
//
// A copy to pageable memory costs 0.4 ms from 1 MB on and runs at 14 GB/s on
// an MI355X host; to pinned memory 54 GB/s are possible.  So kernels write
// results straight into a pinned block (a queued copy of 64 bytes takes 27 us,
// a kernel 5), rods interleaved on their way, and the host copies them on: all
// at once if they fit, else in chunks, one while the next arrive, and with a
// few threads where the caller's memory is so large that its first touch (a
// page fault per 4 KB) is what takes the time.  500,000 rods (16 MB): 5.4 ->
// 0.66 ms; a network of 1.5 M entries (26 MB) 1.8 -> 1.1.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <chrono>
#include <cstring>
#include <string>
#include <system_error>
#include <thread>

#include "nf_host.h"

namespace nf {

namespace {

constexpr size_t PIN_SMALL = 256u << 10, PIN_LARGE = 8u << 20;
constexpr int SLOTS = 8;                       // chunks of the large block
constexpr size_t THREADS_FROM = 8u << 20;      // bytes from which helpers copy
constexpr int HELPERS = 4;
constexpr size_t PLAIN_TO = 768u << 10;        // bytes of one result up to which a plain copy is quicker

// The handle's pinned block, at least `bytes` of it (at most PIN_LARGE); null
// if the host has no pinned memory left.
char* pin_block(nf_handle* h, size_t bytes) {
  if (h->pin && h->pin_bytes >= bytes) return h->pin;
  const size_t want = bytes <= PIN_SMALL ? PIN_SMALL : PIN_LARGE;
  char* p = nullptr;
  if (hipHostMalloc((void**)&p, want, hipHostMallocDefault) != hipSuccess) {
    (void)hipGetLastError();
    return nullptr;
  }
  if (h->pin) (void)hipHostFree(h->pin);
  h->pin = p;
  h->pin_bytes = want;
  return p;
}

bool pin_events(nf_handle* h) {
  for (auto& e : h->pin_ev)
    if (!e && hipEventCreateWithFlags(&e, hipEventDisableTiming) != hipSuccess) {
      (void)hipGetLastError();
      return false;
    }
  return true;
}

struct Piece {
  char* dst;
  size_t part, off, bytes;
};

// issue(part, offset, bytes, to) queues the part's bytes [offset, offset +
// bytes) into pinned memory at `to`.  Returns false, with nothing queued, where
// there is no pinned memory.
template <class Issue>
bool staged(nf_handle* h, const HostPart* parts, size_t n_parts, Issue issue, hipError_t* out) {
  *out = hipSuccess;
  size_t total = 0, padded = 0;
  for (size_t i = 0; i < n_parts; ++i) {
    total += parts[i].bytes;
    padded += (parts[i].bytes + 255) & ~(size_t)255;
  }
  if (total == 0) {
    *out = sync_stream(h->stream, "copy to the host");
    return true;
  }
  if (padded <= PIN_SMALL) {
    char* pin = pin_block(h, padded);
    if (!pin) return false;
    hipError_t e = hipSuccess;
    size_t at = 0;
    for (size_t i = 0; i < n_parts && e == hipSuccess; ++i) {
      if (parts[i].bytes) e = issue(i, 0, parts[i].bytes, pin + at);
      at += (parts[i].bytes + 255) & ~(size_t)255;
    }
    const hipError_t w = sync_stream(h->stream, "copy to the host");
    *out = e != hipSuccess ? e : w;
    if (*out != hipSuccess) return true;
    at = 0;
    for (size_t i = 0; i < n_parts; ++i) {
      if (parts[i].bytes) std::memcpy(parts[i].dst, pin + at, parts[i].bytes);
      at += (parts[i].bytes + 255) & ~(size_t)255;
    }
    return true;
  }
  char* pin = pin_block(h, PIN_LARGE);
  if (!pin || !pin_events(h)) return false;
  const size_t unit = 64u << 10;
  const size_t chunk = std::min(std::max((total / SLOTS + unit - 1) / unit * unit, unit), PIN_LARGE / SLOTS);
  uint64_t n = 0;
  for (size_t i = 0; i < n_parts; ++i) n += (parts[i].bytes + chunk - 1) / chunk;
  auto piece = [&](uint64_t c) {
    size_t i = 0;
    for (;; ++i) {
      const uint64_t k = (parts[i].bytes + chunk - 1) / chunk;
      if (c < k) break;
      c -= k;
    }
    const size_t off = (size_t)c * chunk;
    return Piece{(char*)parts[i].dst + off, i, off, std::min(chunk, parts[i].bytes - off)};
  };
  // chunk c lives in slot c % SLOTS; copied[slot] = 1 + the last chunk copied out of it
  std::atomic<uint64_t> copied[SLOTS], ready{0}, next{0};
  std::atomic<bool> stop{false};
  for (auto& c : copied) c.store(0);
  auto copy_out = [&](uint64_t c) {
    const Piece p = piece(c);
    std::memcpy(p.dst, pin + (c % SLOTS) * chunk, p.bytes);
    copied[c % SLOTS].store(c + 1, std::memory_order_release);
  };
  std::thread helper[HELPERS];
  int helpers = 0;
  if (total >= THREADS_FROM) {
    auto work = [&]() {
      for (;;) {
        const uint64_t c = next.fetch_add(1);
        if (c >= n) return;
        while (ready.load(std::memory_order_acquire) <= c) {
          if (stop.load()) return;
          std::this_thread::yield();
        }
        copy_out(c);
      }
    };
    try {
      for (; helpers < HELPERS; ++helpers) helper[helpers] = std::thread(work);
    } catch (const std::system_error&) {  // no more threads: those that started do
    }
  }
  hipError_t e = hipSuccess;
  uint64_t issued = 0;
  for (uint64_t c = 0; c < n && e == hipSuccess; ++c) {
    for (; issued < n && issued < c + SLOTS; ++issued) {
      const uint64_t slot = issued % SLOTS;
      if (issued >= SLOTS && copied[slot].load(std::memory_order_acquire) != issued - SLOTS + 1) break;
      const Piece p = piece(issued);
      e = issue(p.part, p.off, p.bytes, pin + slot * chunk);
      if (e == hipSuccess) e = hipEventRecord(h->pin_ev[slot], h->stream);
      if (e != hipSuccess) break;
    }
    if (e != hipSuccess) break;
    if (issued <= c) {  // its slot is still being copied out by a helper
      std::this_thread::yield();
      --c;
      continue;
    }
    e = sync_event(h->pin_ev[c % SLOTS], "copy to the host");
    if (e != hipSuccess) break;
    ready.store(c + 1, std::memory_order_release);
    if (helpers == 0) copy_out(c);
  }
  if (e != hipSuccess) stop.store(true);
  for (int k = 0; k < helpers; ++k) helper[k].join();
  if (e != hipSuccess) (void)sync_stream(h->stream, "copy to the host");
  *out = e;
  return true;
}

// The handle's device for the current scope (a caller may have another one
// current; copies had not minded).
struct OnDevice {
  int before = 0;
  bool changed = false;
  explicit OnDevice(int device) {
    if (hipGetDevice(&before) == hipSuccess && before != device) changed = hipSetDevice(device) == hipSuccess;
  }
  ~OnDevice() {
    if (changed) (void)hipSetDevice(before);
  }
};

}  // namespace

namespace {

hipError_t plain(const HostPart* parts, size_t n_parts) {
  hipError_t e = hipSuccess;
  for (size_t i = 0; i < n_parts && e == hipSuccess; ++i)
    if (parts[i].bytes) e = hipMemcpy(parts[i].dst, parts[i].src, parts[i].bytes, hipMemcpyDeviceToHost);
  return e;
}

}  // namespace

hipError_t to_host(nf_handle* h, const HostPart* parts, size_t n_parts) {
  std::lock_guard<std::mutex> lock(h->pin_mu);
  OnDevice on(h->device);
  hipError_t e = hipSuccess;
  const bool done = staged(h, parts, n_parts, [&](size_t i, size_t off, size_t bytes, char* to) {
    launch_to_pinned((const char*)parts[i].src + off, bytes, to, h->stream);
    return hipGetLastError();
  }, &e);
  if (done) return e;
  e = sync_stream(h->stream, "copy to the host");
  return e == hipSuccess ? plain(parts, n_parts) : e;
}

// A plain copy of one short array is back sooner than a staged one where nothing
// has been queued.  Staged and plain, into memory in use / never touched: 72
// bytes 28 and 13 us; 24 KB 25 / 28 and 28 / 32; 164 KB 28 / 60 and 16 / 43; 310 KB
// 42 / 80 and 23 / 74; 960 KB 68 / 219 and 49 / 211; 2.2 MB 84 / 451 and 132 /
// 586.  Several arrays share the staging: four of 480 KB together 75 / 134 and
// 71 / 150.  Behind kernels and device copies of the same call it had cost 30 us
// (nf_reduce of 200,000 rods 290 -> 325).
hipError_t results_to_host(nf_handle* h, const HostPart* parts, size_t n_parts) {
  size_t some = 0, total = 0;
  for (size_t i = 0; i < n_parts; ++i) {
    some += parts[i].bytes ? 1 : 0;
    total += parts[i].bytes;
  }
  if (some == 1 && total <= PLAIN_TO && hipStreamQuery(h->stream) == hipSuccess) {
    std::lock_guard<std::mutex> lock(h->pin_mu);
    OnDevice on(h->device);
    return plain(parts, n_parts);
  }
  return to_host(h, parts, n_parts);
}

hipError_t rods_to_host(nf_handle* h, const float4* P, const float4* D, uint32_t n, float* rods) {
  std::lock_guard<std::mutex> lock(h->pin_mu);
  OnDevice on(h->device);
  const size_t rod = 8 * sizeof(float);
  const HostPart part = {rods, nullptr, n * rod};
  hipError_t e = hipSuccess;
  const bool done = staged(h, &part, 1, [&](size_t, size_t off, size_t bytes, char* to) {
    launch_pack_rods(P + off / rod, D + off / rod, (uint32_t)(bytes / rod), (float4*)to, h->stream);
    return hipGetLastError();
  }, &e);
  if (done) return e;
  constexpr uint32_t STEP = 1024;
  float4 p[STEP], d[STEP];
  e = sync_stream(h->stream, "copy to the host");
  for (uint32_t b = 0; b < n && e == hipSuccess; b += STEP) {
    const uint32_t k = std::min(STEP, n - b);
    e = hipMemcpy(p, P + b, sizeof(float4) * k, hipMemcpyDeviceToHost);
    if (e == hipSuccess) e = hipMemcpy(d, D + b, sizeof(float4) * k, hipMemcpyDeviceToHost);
    for (uint32_t i = 0; i < k && e == hipSuccess; ++i) {
      const float r[8] = {p[i].x, p[i].y, p[i].z, d[i].x, d[i].y, d[i].z, 2.0f * p[i].w, d[i].w};
      std::memcpy(rods + 8 * ((size_t)b + i), r, sizeof(r));
    }
  }
  return e;
}

hipError_t rods_to_device(nf_handle* h, const float* rods, uint32_t n, float4* P, float4* D) {
  if (n == 0) return hipSuccess;
  std::lock_guard<std::mutex> lock(h->pin_mu);
  OnDevice on(h->device);
  const size_t rod = 8 * sizeof(float);
  // slots of the block in turn, filled while the one before is on its way
  char* pin = pin_block(h, n * rod <= PIN_SMALL ? n * rod : PIN_LARGE);
  float4 stack[256];
  const bool piped = pin && pin_events(h);
  const size_t slots = h->pin_bytes > PIN_SMALL ? SLOTS : 1;
  const uint32_t step = piped ? (uint32_t)(h->pin_bytes / slots / rod) : 128u;
  hipError_t e = sync_stream(h->stream, "copy from the host");
  uint64_t k = 0;
  for (uint32_t b = 0; b < n && e == hipSuccess; b += step, ++k) {
    const uint32_t c = std::min(step, n - b);
    const size_t slot = k % slots;
    float4* p = piped ? (float4*)(pin + slot * (h->pin_bytes / slots)) : stack;
    float4* d = p + step;
    if (piped && k >= slots) e = sync_event(h->pin_ev[slot], "copy from the host");
    if (e != hipSuccess) break;
    for (uint32_t i = 0; i < c; ++i) {
      const float* r = rods + 8 * ((size_t)b + i);
      p[i] = make_float4(r[0], r[1], r[2], 0.5f * r[6]);
      d[i] = make_float4(r[3], r[4], r[5], r[7]);
    }
    e = hipMemcpyAsync(P + b, p, sizeof(float4) * c, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess) e = hipMemcpyAsync(D + b, d, sizeof(float4) * c, hipMemcpyHostToDevice, h->stream);
    if (e == hipSuccess && piped) e = hipEventRecord(h->pin_ev[slot], h->stream);
    if (e == hipSuccess && !piped) e = sync_stream(h->stream, "copy from the host");
  }
  const hipError_t w = sync_stream(h->stream, "copy from the host");
  return e != hipSuccess ? e : w;
}

HostScalars* host_scalars(nf_handle* h) {
  if (!h->scal) {
    void* p = nullptr;
    h->scal_pinned = hipHostMalloc(&p, sizeof(HostScalars), hipHostMallocDefault) == hipSuccess;
    if (!h->scal_pinned) (void)hipGetLastError();
    h->scal = h->scal_pinned ? (HostScalars*)p : new HostScalars();
  }
  return h->scal;
}

hipError_t scalars_to_host(nf_handle* h, void* dst, const void* src, size_t bytes) {
  if (!h->scal_pinned) return hipMemcpyAsync(dst, src, bytes, hipMemcpyDeviceToHost, h->stream);
  launch_to_pinned(src, bytes, dst, h->stream);
  return hipGetLastError();
}

void release_pinned(nf_handle* h) {
  for (auto& e : h->pin_ev)
    if (e) (void)hipEventDestroy(e);
  if (h->pin) (void)hipHostFree(h->pin);
  if (h->scal_pinned)
    (void)hipHostFree(h->scal);
  else
    delete h->scal;
}

}  // namespace nf
