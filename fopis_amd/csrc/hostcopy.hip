// Copies between the caller's pageable arrays and the device.
//
// A pageable hipMemcpy of 139 MB (one field at 257^3 nodes) reached 10 GB/s
// into a fresh array and 17 GB/s into a touched one, one thread moving the
// bytes between the runtime's staging and the caller's pages (and taking the
// page faults). Here a few threads each keep two pinned chunks in flight on the
// stream and move them: 43 GB/s into a fresh array (3.2 ms instead of 13.4), 42
// GB/s to the device, where the link is the bound. The chunks cross the link by
// a kernel: hipMemcpyAsync took 3.7 ms in some processes and 12.0 ms in others
// or at other times of one (11.6 GB/s, whichever engine it was given).
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
// From here on the threads are faster than a plain copy (into a fresh array
// 4.6 MB: 0.42 ms for 0.48, 12 MB 0.60 for 1.37; to the device 18 MB: 0.64 for
// 0.52, 35 MB 0.96 for 1.21): they cost 0.2 ms to start.
constexpr size_t kLeastOut = (size_t)4 << 20, kLeastIn = (size_t)24 << 20;
constexpr size_t kLeastChunk = (size_t)512 << 10;
constexpr int kMostThreads = 8;

// A chunk's place in its slot: where it has its device address modulo 16, so
// that both sides take 16-byte accesses.
constexpr size_t kSlot = kChunk + 64;
inline char* in_slot(char* slot, const char* dev) { return slot + (reinterpret_cast<uintptr_t>(dev) & 15); }

// The pinned chunks: one block of 32 MB per process, made by the first large
// copy (a copy with a block of its own took 12 ms), used by one copy at a time
// (another goes the plain way meanwhile), kept while a context lives and given
// back with the last one.
std::mutex g_mu;
char* g_pin = nullptr;
int g_contexts = 0;
bool g_busy = false;

struct Lease {
  char* p = nullptr;
  Lease() {
    std::lock_guard<std::mutex> lk(g_mu);
    if (g_busy || g_contexts == 0) return;
    if (!g_pin && hipHostMalloc(reinterpret_cast<void**>(&g_pin), (size_t)kMostThreads * 2 * kSlot,
                                hipHostMallocPortable | hipHostMallocCoherent) != hipSuccess) {
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

// `bytes` bytes between device memory and a pinned slot, both at the same
// address modulo 16: the ends byte by byte, the rest in 16-byte pieces, a
// wavefront's 1 KB apart.
constexpr int kMoveBlocks = 64;
__global__ __launch_bounds__(256) void k_move(char* __restrict__ to, const char* __restrict__ from, uint32_t bytes) {
  const uint32_t head = min((uint32_t)(-reinterpret_cast<uintptr_t>(from) & 15u), bytes);
  const uint32_t n16 = (bytes - head) / 16, tail = head + 16 * n16;
  const uint4* f = reinterpret_cast<const uint4*>(from + head);
  uint4* t = reinterpret_cast<uint4*>(to + head);
  const uint32_t step = gridDim.x * 256;
  uint32_t i = blockIdx.x * 256 + threadIdx.x;
  for (; i + 3 * step < n16; i += 4 * step) {
    const uint4 a = f[i], b = f[i + step], c = f[i + 2 * step], d = f[i + 3 * step];
    t[i] = a;
    t[i + step] = b;
    t[i + 2 * step] = c;
    t[i + 3 * step] = d;
  }
  for (; i < n16; i += step) t[i] = f[i];
  if (blockIdx.x == 0 && threadIdx.x < 32) {
    const uint32_t e = threadIdx.x < 16 ? threadIdx.x : tail + threadIdx.x - 16;
    if (threadIdx.x < 16 ? e < head : e < bytes) to[e] = from[e];
  }
}

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
    char* slot = pin + (size_t)s * kSlot;
    if (busy[s]) {
      const Chunk& c = chunks[idx[s]];
      good = ok(hipEventSynchronize(ev[s]));
      if (good && to_host) std::memcpy(c.host, in_slot(slot, c.dev), c.bytes);
      busy[s] = false;
    }
    const size_t i = good && err.load() == (int)hipSuccess ? next.fetch_add(1) : chunks.size();
    if (i < chunks.size()) {
      const Chunk& c = chunks[i];
      idx[s] = i;
      char* at = in_slot(slot, c.dev);
      if (!to_host) std::memcpy(at, c.host, c.bytes);
      k_move<<<kMoveBlocks, 256, 0, st>>>(to_host ? at : c.dev, to_host ? c.dev : at, (uint32_t)c.bytes);
      good = ok(hipGetLastError()) && ok(hipEventRecord(ev[s], st));
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
  if (total < (to_host ? kLeastOut : kLeastIn)) return plain();
  const int cpus = std::max(1, (int)std::thread::hardware_concurrency() / 2);
  // a thread takes two chunks or more where there are enough
  const size_t chunk = std::min(kChunk, std::max(kLeastChunk, (total / (2 * kMostThreads) + 4095) / 4096 * 4096));
  const int nt = (int)std::min<size_t>({(size_t)kMostThreads, (size_t)cpus, total / chunk});
  if (nt < 2) return plain();
  Lease pin;
  if (!pin.p) return plain();
  std::vector<Chunk> chunks;
  for (int q = 0; q < nseg; ++q)
    for (size_t at = 0; at < seg[q].bytes; at += chunk)
      chunks.push_back(Chunk{static_cast<char*>(seg[q].host) + at, static_cast<char*>(seg[q].dev) + at,
                             std::min(chunk, seg[q].bytes - at)});
  int dev = 0;
  FOPIS_HIP(hipGetDevice(&dev));
  std::atomic<size_t> next{0};
  std::atomic<int> err{(int)hipSuccess};
  std::vector<std::thread> th;
  th.reserve(nt);
  try {
    for (int t = 1; t < nt; ++t)
      th.emplace_back(work, std::cref(chunks), std::ref(next), std::ref(err), pin.p + (size_t)t * 2 * kSlot, to_host, st,
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
