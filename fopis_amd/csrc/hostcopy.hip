// Copies between the caller's pageable arrays and the device.
//
// A pageable hipMemcpy of 139 MB (one field at 257^3 nodes) reached 10 GB/s
// into a fresh array and 17 GB/s into a touched one, one thread moving the
// bytes between the runtime's staging and the caller's pages (and taking the
// page faults). Here the calling thread launches the chunks and a few threads
// move them to or from the caller's pages, two pinned slots to a thread: 43 GB/s
// into a fresh array (3.2 ms instead of 13.4), 38 GB/s to the device, where the
// link is the bound. The chunks cross the link by a kernel: hipMemcpyAsync took
// 3.7 ms in some processes and 12.0 ms in others or at other times of one (11.6
// GB/s, whichever engine it was given).
#include <hip/hip_runtime.h>

#include <algorithm>
#include <atomic>
#include <cstring>
#include <exception>
#include <fstream>
#include <limits>
#include <memory>
#include <mutex>
#include <string>
#include <thread>
#include <vector>

#include "fopis_internal.hpp"

namespace fopis {

namespace {

constexpr size_t kChunk = (size_t)2 << 20;
// From here on the threads are faster than a plain copy (2.4 MB out: 0.28 ms for
// 0.55 into fresh arrays, 0.11 for 0.14 into touched ones; 7.8 MB 0.50 for 0.98
// and 0.29 for 0.44; in, 18 MB: 0.59 for 0.52, 35 MB 1.10 for 1.21). A small
// copy takes fewer of them.
constexpr size_t kLeastOut = (size_t)2 << 20, kLeastIn = (size_t)24 << 20;
constexpr size_t kLeastChunk = (size_t)128 << 10, kPerThread = (size_t)1280 << 10;
constexpr int kMostThreads = 8;
// A small copy out takes one chunk per piece and no thread (55 KB: 18 us, where
// hipMemcpyAsync took 17 in some processes and 33 in others; 157 KB: 23 for 17).
constexpr size_t kSmall = (size_t)64 << 10;
constexpr int kSmallSegs = 8;

// A chunk's place in its slot: where it has its device address modulo 16, so
// that both sides take 16-byte accesses.
constexpr size_t kSlot = kChunk + 64;
inline char* in_slot(char* slot, const char* dev) { return slot + (reinterpret_cast<uintptr_t>(dev) & 15); }

// The pinned memory: one block for large copies and one for small ones per
// process, each made by the first copy that wants it, used by one copy at a
// time (another goes the plain way meanwhile), kept while a context lives and
// given back with the last one. The word behind the chunks is Copy::landed.
// The large one starts with kFirst bytes, for copies out of kLeastFirst and more
// by two threads, and becomes 32 MB once the copies have asked for kWorth
// bytes: pinning and touching 32 MB takes 0.6 to 1.6 ms (1 MB 0.04), which a
// program that reads one field and closes its context would not get back. Plain
// 2.6 MB take 160 us, 4.6 MB 285, 7.8 MB 470, 18 MB 1100; through 1 MB 160, 240,
// 370, 770; through 32 MB 115, 190, 270, 520: some 15 us a MB less than through
// 1 MB, so 48 MB of copies save about what the large block costs.
constexpr size_t kFirst = ((size_t)1 << 20) + 64, kLeastFirst = (size_t)4 << 20, kWorth = (size_t)48 << 20;
struct Block {
  size_t first, full;
  char* p = nullptr;
  bool busy = false;
  size_t bytes = 0, asked = 0;
};
std::mutex g_mu;
Block g_large{kFirst, (size_t)kMostThreads * 2 * kSlot + 64};
Block g_small{kSmall + kSmallSegs * 32 + 64, kSmall + kSmallSegs * 32 + 64};
int g_contexts = 0;

struct Lease {
  Block& b;
  char* p = nullptr;
  // a copy of `total` bytes, for which the first size will do or not
  Lease(Block& block, size_t total, bool first_serves) : b(block) {
    std::lock_guard<std::mutex> lk(g_mu);
    if (b.busy || g_contexts == 0) return;
    b.asked = std::min(kWorth, b.asked + std::min(kWorth, total));
    const size_t want = b.asked == kWorth ? b.full : b.first;
    if (b.bytes < b.full && want < b.full && !first_serves) return;
    if (b.bytes < want) {
      drop(b);
      if (hipHostMalloc(reinterpret_cast<void**>(&b.p), want, hipHostMallocPortable | hipHostMallocCoherent) !=
          hipSuccess) {
        b.p = nullptr;
        (void)hipGetLastError();
        return;
      }
      b.bytes = want;
    }
    b.busy = true;
    p = b.p;
  }
  ~Lease() {
    if (!p) return;
    std::lock_guard<std::mutex> lk(g_mu);
    b.busy = false;
    give_back();
  }
  size_t room() const { return (b.bytes - 64) / 16 * 16; }
  uint32_t* word() const { return reinterpret_cast<uint32_t*>(p + room()); }
  static void drop(Block& q) {
    if (q.p) (void)hipHostFree(q.p);
    q.p = nullptr;
    q.bytes = 0;
  }
  static void give_back() {  // with g_mu held
    if (g_contexts > 0) return;
    for (Block* q : {&g_large, &g_small})
      if (!q->busy) {
        drop(*q);
        q->asked = 0;
      }
  }
};

// `bytes` bytes between device memory and a pinned slot, both at the same
// address modulo 16: the ends byte by byte, the rest in 16-byte pieces, a
// wavefront's 1 KB apart. 64 workgroups: 128 took 3.4 ms out and 4.6 in for 139
// MB, 64 3.2 and 3.7.
// A launch first tells the host that the chunks before its own have landed.
constexpr int kMoveBlocks = 64;
__global__ __launch_bounds__(256) void k_move(char* __restrict__ to, const char* __restrict__ from, uint32_t bytes,
                                              uint32_t* landed, uint32_t chunk) {
  if (blockIdx.x == 0 && threadIdx.x == 0) {
    *reinterpret_cast<volatile uint32_t*>(landed) = chunk;
  }
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
  __threadfence_system();  // the next launch announces this chunk
}

__global__ void k_landed(uint32_t* landed, uint32_t chunks) { *reinterpret_cast<volatile uint32_t*>(landed) = chunks; }

// The launches' own status: hipGetLastError would also give what an earlier
// call of this thread left there, its program's or this library's.
hipError_t launch_move(char* to, const char* from, size_t bytes, uint32_t* landed, size_t chunk, size_t blocks,
                       hipStream_t st) {
  uint32_t n = (uint32_t)bytes, k = (uint32_t)chunk;
  void* a[] = {&to, &from, &n, &landed, &k};
  return hipLaunchKernel(reinterpret_cast<const void*>(&k_move), dim3((unsigned)blocks), dim3(256), a, 0, st);
}

hipError_t launch_landed(uint32_t* landed, size_t chunks, hipStream_t st) {
  uint32_t k = (uint32_t)chunks;
  void* a[] = {&landed, &k};
  return hipLaunchKernel(reinterpret_cast<const void*>(&k_landed), dim3(1), dim3(1), a, 0, st);
}

struct Chunk {
  char* host;
  char* dev;
  size_t bytes;
};

// One copy. The calling thread launches the chunks in order and moves bytes
// like the other threads, which make no runtime calls (a thread's first ones
// cost it 0.1 ms; 2.4 MB out took 0.42 ms with them into fresh arrays, 0.28
// without). Chunk i uses slot i % nslots.
struct Copy {
  std::vector<Chunk> chunks;
  std::unique_ptr<std::atomic<uint8_t>[]> moved;  // by a thread, between the caller's array and the slot
  std::atomic<size_t> next{0}, nmoved{0};
  std::atomic<bool> stop{false};
  char* pin = nullptr;
  uint32_t* landed = nullptr;  // chunks whose kernels have ended
  size_t nslots = 0, slot_bytes = 0, launched = 0;
  bool to_host = false;
  hipStream_t st = nullptr;
  hipError_t err = hipSuccess;

  char* slot(size_t i) const { return in_slot(pin + (i % nslots) * slot_bytes, chunks[i].dev); }
  size_t ended() const { return __atomic_load_n(landed, __ATOMIC_ACQUIRE); }

  // launches every chunk that may go (the calling thread)
  void pump() {
    const size_t n = chunks.size();
    while (launched < n && !stop.load()) {
      const size_t i = launched;
      if (to_host ? i >= nslots && !moved[i - nslots].load(std::memory_order_acquire)
                  : !moved[i].load(std::memory_order_acquire))
        return;
      const Chunk& c = chunks[i];
      fail(launch_move(to_host ? slot(i) : c.dev, to_host ? c.dev : slot(i), c.bytes, landed, i, kMoveBlocks, st));
      if (++launched == n) fail(launch_landed(landed, n, st));
    }
  }
  void fail(hipError_t e) {
    if (e == hipSuccess) return;
    if (err == hipSuccess) err = e;
    stop.store(true);
  }
  // waits until ready() (or stop); the calling thread keeps launching meanwhile
  template <class F>
  void wait(bool caller, F ready) {
    for (unsigned k = 1; !ready() && !stop.load(std::memory_order_relaxed); ++k) {
      if (caller) pump();
      if (caller && (k & 0xffff) == 0) {
        const hipError_t e = hipStreamQuery(st);
        if (e != hipErrorNotReady) fail(e);
        if (hipPeekAtLastError() == hipErrorNotReady) (void)hipGetLastError();  // no error of a later launch
      }
      if ((k & 0xff) == 0) std::this_thread::yield();
    }
  }
  void work(bool caller, bool moves) {
    const size_t n = chunks.size();
    if (caller) pump();
    for (size_t i; moves && (i = next.fetch_add(1)) < n;) {
      const Chunk& c = chunks[i];
      if (to_host) {
        wait(caller, [&] { return ended() > i; });
        if (stop.load()) return;
        std::memcpy(c.host, slot(i), c.bytes);
      } else {
        wait(caller, [&] { return i < nslots || ended() > i - nslots; });
        if (stop.load()) return;
        std::memcpy(slot(i), c.host, c.bytes);
      }
      moved[i].store(1, std::memory_order_release);
      nmoved.fetch_add(1);
      if (caller) pump();
    }
    // only the calling thread asks the stream for errors: it goes on until no thread waits for a chunk
    if (caller) wait(true, [&] { return launched == n && nmoved.load() == n; });
  }
};

}  // namespace

// The CPUs that a control group's quota amounts to, rounded down but at least
// one, from the files under `root` (version 2, then 1); without a quota the most.
int quota_cpus(const char* root) {
  double quota = 0.0, period = 0.0;
  std::ifstream v2(std::string(root) + "/cpu.max");
  if (!(v2 >> quota >> period)) {  // ("max" is no number)
    std::ifstream q(std::string(root) + "/cpu/cpu.cfs_quota_us"), p(std::string(root) + "/cpu/cpu.cfs_period_us");
    if (!(q >> quota) || !(p >> period)) quota = 0.0;  // (-1 is none)
  }
  if (!(quota > 0.0 && period > 0.0)) return std::numeric_limits<int>::max();
  return std::max(1, (int)std::min(quota / period, 65536.0));
}

void host_copy_retain() {
  std::lock_guard<std::mutex> lk(g_mu);
  ++g_contexts;
}

void host_copy_release() {
  std::lock_guard<std::mutex> lk(g_mu);
  --g_contexts;
  Lease::give_back();
}

// An array that the runtime knows (pinned by the caller, say) is copied
// directly by a plain copy, faster than through the blocks here: 54 KB out in 9
// us for 18, 2.6 MB in 54 for 115, 139 MB in 2.4 ms for 3.1.
bool known(const HostSeg* seg, int nseg) {
  for (int q = 0; q < nseg; ++q) {
    hipPointerAttribute_t a{};
    if (seg[q].bytes == 0) continue;
    const hipError_t e = hipPointerGetAttributes(&a, seg[q].host);
    if (e == hipSuccess && a.type != hipMemoryTypeUnregistered) return true;
    if (e != hipSuccess && hipPeekAtLastError() == e) (void)hipGetLastError();
  }
  return false;
}

// Copies every segment and returns when the copies are done.
void host_copy(const HostSeg* seg, int nseg, bool to_host, hipStream_t st) {
  size_t total = 0;
  for (int q = 0; q < nseg; ++q) {
    if (seg[q].bytes > 0 && (!seg[q].host || !seg[q].dev)) FOPIS_HIP(hipErrorInvalidValue);  // as a plain copy says
    total += seg[q].bytes;
  }
  auto plain = [&] {
    for (int q = 0; q < nseg; ++q) {
      if (seg[q].bytes == 0) continue;
      FOPIS_HIP(to_host ? hipMemcpyAsync(seg[q].host, seg[q].dev, seg[q].bytes, hipMemcpyDeviceToHost, st)
                        : hipMemcpyAsync(seg[q].dev, seg[q].host, seg[q].bytes, hipMemcpyHostToDevice, st));
    }
    FOPIS_HIP(hipStreamSynchronize(st));
  };
  if (to_host && total > 0 && total <= kSmall && nseg <= kSmallSegs) {
    if (known(seg, nseg)) return plain();
    Lease pin(g_small, 0, true);
    if (!pin.p) return plain();
    char* at[kSmallSegs];
    size_t off = 0;
    hipError_t launched = hipSuccess;
    for (int q = 0; q < nseg; ++q) {
      const char* dev = static_cast<const char*>(seg[q].dev);
      at[q] = in_slot(pin.p + off, dev);
      off += (seg[q].bytes + 31) / 16 * 16;
      if (seg[q].bytes > 0 && launched == hipSuccess)
        launched = launch_move(at[q], dev, seg[q].bytes, pin.word(), 0,
                               std::min<size_t>(kMoveBlocks, seg[q].bytes / 4096 + 1), st);
    }
    // (on an error too: nothing may be in flight when the next copy takes the block)
    const hipError_t ended = hipStreamSynchronize(st);
    FOPIS_HIP(launched);
    FOPIS_HIP(ended);
    for (int q = 0; q < nseg; ++q) std::memcpy(seg[q].host, at[q], seg[q].bytes);
    return;
  }
  if (total < (to_host ? kLeastOut : kLeastIn)) return plain();
  static const int cpus = std::min((int)std::thread::hardware_concurrency(), quota_cpus("/sys/fs/cgroup")) / 2;
  if (cpus < 2 || known(seg, nseg)) return plain();
  Lease pin(g_large, total, to_host && total >= kLeastFirst);
  if (!pin.p) return plain();
  const int nt = pin.b.bytes < pin.b.full ? 2
                                          : (int)std::min<size_t>({(size_t)kMostThreads, (size_t)cpus,
                                                                   std::max<size_t>(2, total / kPerThread)});
  const size_t slot = std::min(kSlot, pin.room() / (2 * (size_t)nt) / 64 * 64);
  const size_t chunk = std::min((slot - 64) / 4096 * 4096,
                                std::max(kLeastChunk, (total / (3 * (size_t)nt) + 4095) / 4096 * 4096));
  Copy c;
  for (int q = 0; q < nseg; ++q)
    for (size_t at = 0; at < seg[q].bytes; at += chunk)
      c.chunks.push_back(Chunk{static_cast<char*>(seg[q].host) + at, static_cast<char*>(seg[q].dev) + at,
                               std::min(chunk, seg[q].bytes - at)});
  c.moved.reset(new std::atomic<uint8_t>[c.chunks.size()]);
  for (size_t i = 0; i < c.chunks.size(); ++i) c.moved[i].store(0);
  c.pin = pin.p;
  c.landed = pin.word();
  *c.landed = 0;
  c.nslots = (size_t)nt * 2;
  c.slot_bytes = slot;
  c.to_host = to_host;
  c.st = st;
  std::vector<std::thread> th;
  th.reserve(nt);
  // The threads wait for this copy alone, not through what the stream still has
  // to do: they start on an idle stream, or when the first chunk has come out
  // (the others follow it while they start).
  if (to_host) {
    c.pump();
    c.wait(true, [&] { return c.ended() > 0; });
  } else {
    c.fail(hipStreamSynchronize(st));
  }
  try {
    for (int t = to_host ? 1 : 0; t < nt && !c.stop.load(); ++t) th.emplace_back([&c] { c.work(false, true); });
  } catch (const std::exception&) {
    // no thread or no memory for one: those that started, and this one, take every chunk
  }
  // (on the way in the caller only launches: no chunk waits while it moves one)
  c.work(true, to_host || th.empty());
  for (auto& t : th) t.join();
  // (on an error too: nothing may be in flight when the next copy takes the block)
  const hipError_t e = hipStreamSynchronize(st);
  FOPIS_HIP(c.err);
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
