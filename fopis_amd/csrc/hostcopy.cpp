// Copies between the caller's pageable arrays and the device.
//
// A pageable hipMemcpy of 139 MB (one field at 257^3 nodes) reached 10 GB/s
// into a fresh array and 17 GB/s into a touched one, one thread moving the
// bytes between the runtime's staging and the caller's pages (and taking the
// page faults). Here a few threads each keep two pinned 2 MB chunks in flight
// on the stream and move them: 37 GB/s into a fresh array (3.9 ms instead of
// 13.7), 38 GB/s otherwise and to the device, where the link is the bound.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <mutex>
#include <system_error>
#include <thread>
#include <vector>

#include "fopis_internal.hpp"

namespace fopis {

namespace {

constexpr size_t kChunk = (size_t)2 << 20;
// Below this one thread is as fast (8 MB: 0.44 ms).
constexpr size_t kLeast = (size_t)8 << 20;
constexpr int kMostThreads = 8;

// The pinned chunks: one block of 32 MB per process, made by the first large
// copy (its pages cost 8 ms once, more than a copy saves), used by one copy at
// a time (another goes the plain way meanwhile), kept while a context lives and
// given back with the last one.
std::mutex g_mu;
char* g_pin = nullptr;
int g_contexts = 0;
bool g_busy = false;

struct Lease {
  char* p = nullptr;
  Lease() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_busy || g_contexts == 0) return;
    if (!g_pin && hipHostMalloc(reinterpret_cast<void**>(&g_pin), (size_t)kMostThreads * 2 * kChunk,
                                hipHostMallocPortable) != hipSuccess) {
      g_pin = nullptr;
      (void)hipGetLastError();
      return;
    }
    g_busy = true;
    p = g_pin;
  }
  ~Lease() {
    if (!p) return;
    std::lock_guard<std::mutex> lk(g_mu);
    g_busy = false;
    give_back();
  }
  static void give_back() {  // with g_mu held
    if (g_contexts > 0 || g_busy || !g_pin) return;
    (void)hipHostFree(g_pin);
    g_pin = nullptr;
  }
};

struct Chunk {
  char* host;
  char* dev;
  size_t bytes;
};

// One worker: up to two chunks in flight, in the order they are claimed.
void work(const std::vector<Chunk>& chunks, std::atomic<size_t>& next, std::atomic<int>& err, char* pin, bool to_host,
          hipStream_t st, int dev) {
  hipEvent_t ev[2] = {nullptr, nullptr};
  size_t idx[2] = {0, 0};
  bool busy[2] = {false, false};
  auto ok = [&](hipError_t e) {
    if (e != hipSuccess) {
      int none = (int)hipSuccess;
      err.compare_exchange_strong(none, (int)e);
    }
    return e == hipSuccess;
  };
  bool good = ok(hipSetDevice(dev));
  for (auto& e : ev) good = good && ok(hipEventCreateWithFlags(&e, hipEventDisableTiming));
  int s = 0;
  // slot s: finish what it holds, then the next chunk; ends when both are empty
  while (good) {
    char* slot = pin + (size_t)s * kChunk;
    if (busy[s]) {
      good = ok(hipEventSynchronize(ev[s]));
      if (good && to_host) std::memcpy(chunks[idx[s]].host, slot, chunks[idx[s]].bytes);
      busy[s] = false;
    }
    const size_t i = good && err.load() == (int)hipSuccess ? next.fetch_add(1) : chunks.size();
    if (i < chunks.size()) {
      const Chunk& c = chunks[i];
      idx[s] = i;
      if (!to_host) std::memcpy(slot, c.host, c.bytes);
      good = ok(to_host ? hipMemcpyAsync(slot, c.dev, c.bytes, hipMemcpyDeviceToHost, st)
                        : hipMemcpyAsync(c.dev, slot, c.bytes, hipMemcpyHostToDevice, st)) &&
             ok(hipEventRecord(ev[s], st));
      busy[s] = true;
    } else if (!busy[s ^ 1]) {
      break;
    }
    s ^= 1;
  }
  for (auto& e : ev)
    if (e) (void)hipEventDestroy(e);
}

}  // namespace

void host_copy_retain() {
  std::lock_guard<std::mutex> lk(g_mu);
  ++g_contexts;
}

void host_copy_release() {
  std::lock_guard<std::mutex> lk(g_mu);
  --g_contexts;
  Lease::give_back();
}

// Copies every segment and returns when the copies are done.
void host_copy(const HostSeg* seg, int nseg, bool to_host, hipStream_t st) {
  size_t total = 0;
  for (int q = 0; q < nseg; ++q) total += seg[q].bytes;
  auto plain = [&] {
    for (int q = 0; q < nseg; ++q) {
      if (seg[q].bytes == 0) continue;
      FOPIS_HIP(to_host ? hipMemcpyAsync(seg[q].host, seg[q].dev, seg[q].bytes, hipMemcpyDeviceToHost, st)
                        : hipMemcpyAsync(seg[q].dev, seg[q].host, seg[q].bytes, hipMemcpyHostToDevice, st));
    }
    FOPIS_HIP(hipStreamSynchronize(st));
  };
  if (total < kLeast) return plain();
  const int cpus = std::max(1, (int)std::thread::hardware_concurrency() / 2);
  const int nt = (int)std::min<size_t>({(size_t)kMostThreads, (size_t)cpus, total / (2 * kChunk)});
  if (nt < 2) return plain();
  Lease pin;
  if (!pin.p) return plain();
  std::vector<Chunk> chunks;
  for (int q = 0; q < nseg; ++q)
    for (size_t at = 0; at < seg[q].bytes; at += kChunk)
      chunks.push_back(Chunk{static_cast<char*>(seg[q].host) + at, static_cast<char*>(seg[q].dev) + at,
                             std::min(kChunk, seg[q].bytes - at)});
  int dev = 0;
  FOPIS_HIP(hipGetDevice(&dev));
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  std::vector<std::thread> th;
  th.reserve(nt);
  try {
    for (int t = 1; t < nt; ++t)
      th.emplace_back(work, std::cref(chunks), std::ref(next), std::ref(err), pin.p + (size_t)t * 2 * kChunk, to_host, st,
                      dev);
  } catch (const std::system_error&) {
    // fewer threads than asked for: those that started, and this one, take every chunk
  }
  work(chunks, next, err, pin.p, to_host, st, dev);
  for (auto& t : th) t.join();
  // (on an error too: nothing may be in flight when the next copy takes the block)
  const hipError_t e = hipStreamSynchronize(st);
  FOPIS_HIP((hipError_t)err.load());
  FOPIS_HIP(e);
}

void copy_out(void* host, const void* dev, size_t bytes, hipStream_t st) {
  const HostSeg s{host, const_cast<void*>(dev), bytes};
  host_copy(&s, 1, true, st);
}

void copy_in(void* dev, const void* host, size_t bytes, hipStream_t st) {
  const HostSeg s{const_cast<void*>(host), dev, bytes};
  host_copy(&s, 1, false, st);
}

}  // namespace fopis
