// A HIP runtime without a device, preloaded in front of the real one so that
// libfopis_hip.so's host code runs on the CPU and meets errors that a GPU test
// must not provoke: device memory is host memory, launches are logged and do
// nothing, except that host copies' kernels move their bytes and a solve's
// last kernel reports its cycles. fake_* (C linkage) steer it.
#include <dlfcn.h>
#include <hip/hip_runtime_api.h>

#include <chrono>
#include <condition_variable>
#include <cstdlib>
#include <cstring>
#include <deque>
#include <exception>
#include <map>
#include <mutex>
#include <new>
#include <string>
#include <thread>
#include <vector>

namespace {

std::mutex mu;
std::map<const void*, std::string> kernels;
std::map<const void*, void*> symbols;
std::map<char*, size_t> pinned;
std::map<std::pair<const void*, int>, size_t> granted;  // LDS beyond 64 KB, by kernel and device
std::string log_text;
int fail_malloc = -1, fail_launch = -1, fail_thread = -1, device = 0, cycles = 5, delay_ms = 0;
bool broken = false;
int break_after = -1;
thread_local hipError_t last = hipSuccess;

struct Config {
  dim3 grid, block;
  size_t lds;
  hipStream_t st;
};
thread_local std::vector<Config> configs;

hipError_t ret(hipError_t e) {
  if (e != hipSuccess) last = e;
  return e;
}

void note(const std::string& s) {
  std::lock_guard<std::mutex> lk(mu);
  log_text += s + "\n";
}

// What a launch or a graph does when the stream reaches it.
struct Op {
  char* to = nullptr;
  const char* from = nullptr;
  uint32_t bytes = 0;
  uint32_t* landed = nullptr;
  uint32_t chunk = 0;
  bool last_busy = false;
  char* words = nullptr;  // a solve's: done, confirmed, cycles, updates, pair passes, two residuals
  void run() const {
    if (landed) __atomic_store_n(landed, chunk, __ATOMIC_RELEASE);
    if (to) std::memcpy(to, from, bytes);
    if (words) {
      const int32_t w[5] = {1, 1, cycles, 0, 0};
      const double r[2] = {0.0, 1.0};
      std::memcpy(words, w, sizeof(w));
      std::memcpy(words + 24, r, sizeof(r));
    }
  }
};

// The one queue: launches run in order after a delay, when there is one.
// (never destroyed: its thread waits on it until the process ends)
auto& queue = *new std::deque<Op>;
auto& cv = *new std::condition_variable;
auto& qmu = *new std::mutex;
bool worker = false, busy = false;

void work() {
  std::unique_lock<std::mutex> lk(qmu);
  for (;;) {
    cv.wait(lk, [] { return !queue.empty(); });
    const Op o = queue.front();
    lk.unlock();
    std::this_thread::sleep_for(std::chrono::milliseconds(delay_ms));
    o.run();
    if (o.last_busy) busy = false;
    lk.lock();
    queue.pop_front();
    cv.notify_all();
  }
}

void submit(const Op& o) {
  if (break_after >= 0 && break_after-- == 0) broken = true;
  if (broken) return;
  if (!delay_ms) return o.run();
  std::lock_guard<std::mutex> lk(qmu);
  if (!worker) std::thread(work).detach();
  worker = true;
  queue.push_back(o);
  cv.notify_all();
}

struct Graph {
  size_t nodes = 0;
  std::vector<Op> ops;
};
thread_local Graph* capturing = nullptr;

}  // namespace

extern "C" {

void fake_fail_malloc(int k) { fail_malloc = k; }  // the k-th device allocation from now fails (0: the next)
void fake_fail_launch(int k) { fail_launch = k; }
void fake_fail_thread(int k) { fail_thread = k; }  // starting the k-th thread from now throws std::bad_alloc
int fake_pending() {
  std::lock_guard<std::mutex> lk(qmu);
  return (int)queue.size();
}
void fake_break_stream(int on) { broken = on != 0; }  // nothing launched runs, waits and queries return an error
void fake_break_stream_after(int k) { break_after = k; }  // once k more have run
void fake_delay(int ms) { delay_ms = ms; }
void fake_busy() {  // work of the stream that is not a copy's
  busy = true;
  Op o;
  o.last_busy = true;
  submit(o);
}
void fake_cycles(int n) { cycles = n; }
void fake_set_device(int d) { device = d; }
void fake_log_clear() {
  std::lock_guard<std::mutex> lk(mu);
  log_text.clear();
}
const char* fake_log() { return log_text.c_str(); }

// The library's copy of several arrays, called directly.
struct Seg {
  void *host, *dev;
  size_t bytes;
};
int fake_copy(void (*host_copy)(const Seg*, int, bool, hipStream_t), const Seg* s, int n, int out) {
  try {
    host_copy(s, n, out != 0, nullptr);
    return 0;
  } catch (const std::exception&) {
    return 1;
  }
}

// std::thread's start
void start_thread(void* self, void* state, void (*depend)()) __asm__(
    "_ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE");
void start_thread(void* self, void* state, void (*depend)()) {
  static const auto real = reinterpret_cast<void (*)(void*, void*, void (*)())>(
      dlsym(RTLD_NEXT, "_ZNSt6thread15_M_start_threadESt10unique_ptrINS_6_StateESt14default_deleteIS1_EEPFvvE"));
  note("thread " + std::string(busy ? "busy" : "idle"));
  if (fail_thread >= 0 && fail_thread-- == 0) throw std::bad_alloc();
  real(self, state, depend);
}

void** __hipRegisterFatBinary(const void*) {
  static void* h = nullptr;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  kernels[f] = name;
}
void __hipRegisterVar(void**, void* var, char*, char*, int, size_t size, int, int) {
  symbols[var] = std::calloc(1, size);
}
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t lds, hipStream_t st) {
  configs.push_back({g, b, lds, st});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3* g, dim3* b, size_t* lds, hipStream_t* st) {
  const Config c = configs.back();
  configs.pop_back();
  *g = c.grid;
  *b = c.block;
  *lds = c.lds;
  *st = c.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void* f, dim3 g, dim3, void** a, size_t lds, hipStream_t) {
  {
    std::lock_guard<std::mutex> lk(mu);
    if (lds > 65536 && lds > granted[{f, device}]) return ret(hipErrorInvalidValue);
  }
  if (fail_launch >= 0 && fail_launch-- == 0) return ret(hipErrorLaunchOutOfResources);
  if ((uint64_t)g.x * g.y * g.z >= ((uint64_t)1 << 32)) return ret(hipErrorInvalidConfiguration);
  const std::string& name = kernels[f];
  note("launch " + name + " " + std::to_string(g.x) + " " + std::to_string(g.y) + " " + std::to_string(g.z));
  Op o;
  if (name.find("6k_move") != std::string::npos) {
    o.to = *static_cast<char**>(a[0]);
    o.from = *static_cast<const char**>(a[1]);
    o.bytes = *static_cast<uint32_t*>(a[2]);
    o.landed = *static_cast<uint32_t**>(a[3]);
    o.chunk = *static_cast<uint32_t*>(a[4]);
  } else if (name.find("8k_landed") != std::string::npos) {
    o.landed = *static_cast<uint32_t**>(a[0]);
    o.chunk = *static_cast<uint32_t*>(a[1]);
  } else if (name.find("12k_norm_final") != std::string::npos) {
    o.words = *static_cast<char**>(a[6]);
  }
  if (capturing) {
    ++capturing->nodes;
    if (o.words) capturing->ops.push_back(o);
    return hipSuccess;
  }
  if (o.to || o.landed || o.words) submit(o);
  return hipSuccess;
}

hipError_t hipMalloc(void** p, size_t n) {
  if (fail_malloc >= 0 && fail_malloc-- == 0) {
    note("malloc failed " + std::to_string(n));
    return ret(hipErrorOutOfMemory);
  }
  note("malloc " + std::to_string(n));
  *p = std::calloc(1, n ? n : 1);
  return *p ? hipSuccess : ret(hipErrorOutOfMemory);
}
hipError_t hipFree(void* p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void** p, size_t n, unsigned) {
  note("pin " + std::to_string(n));
  *p = std::calloc(1, n);
  std::lock_guard<std::mutex> lk(mu);
  pinned[static_cast<char*>(*p)] = n;
  return hipSuccess;
}
hipError_t hipPointerGetAttributes(hipPointerAttribute_t* a, const void* p) {
  *a = {};
  std::lock_guard<std::mutex> lk(mu);
  auto it = pinned.upper_bound(static_cast<char*>(const_cast<void*>(p)));
  const bool in = it != pinned.begin() && p < (--it)->first + it->second;
  a->type = in ? hipMemoryTypeHost : hipMemoryTypeUnregistered;
  return hipSuccess;
}
hipError_t hipHostFree(void* p) {
  {
    std::lock_guard<std::mutex> lk(mu);
    pinned.erase(static_cast<char*>(p));
  }
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemGetInfo(size_t* f, size_t* t) {
  *f = *t = (size_t)16 << 30;
  return hipSuccess;
}
static hipError_t sync() {
  if (broken) return ret(hipErrorLaunchFailure);
  std::unique_lock<std::mutex> lk(qmu);
  cv.wait(lk, [] { return queue.empty(); });
  return hipSuccess;
}
hipError_t hipMemcpyAsync(void* d, const void* s, size_t n, hipMemcpyKind, hipStream_t) {
  if (!d || !s) return ret(hipErrorInvalidValue);
  const hipError_t e = sync();
  note("memcpy " + std::to_string(n));
  if (e == hipSuccess) std::memcpy(d, s, n);
  return e;
}
hipError_t hipMemcpy(void* d, const void* s, size_t n, hipMemcpyKind k) { return hipMemcpyAsync(d, s, n, k, nullptr); }
hipError_t hipMemsetAsync(void* d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return hipSuccess;
}
hipError_t hipMemset(void* d, int v, size_t n) { return hipMemsetAsync(d, v, n, nullptr); }

hipError_t hipGetDevice(int* d) {
  *d = device;
  return hipSuccess;
}
hipError_t hipGetDeviceCount(int* n) {
  *n = 2;
  return hipSuccess;
}
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600* p, int) {
  std::memset(p, 0, sizeof(*p));
  std::strcpy(p->name, "none");
  p->sharedMemPerBlock = 163840;
  p->multiProcessorCount = 256;
  return hipSuccess;
}
hipError_t hipFuncSetAttribute(const void* f, hipFuncAttribute, int v) {
  std::lock_guard<std::mutex> lk(mu);
  granted[{f, device}] = (size_t)v;
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void** p, const void* s) {
  *p = symbols[s];
  return *p ? hipSuccess : ret(hipErrorInvalidSymbol);
}
const char* hipGetErrorString(hipError_t e) { return e == hipErrorNotReady ? "not ready" : "error of the fake runtime"; }
hipError_t hipGetLastError() {
  const hipError_t e = last;
  last = hipSuccess;
  return e;
}
hipError_t hipPeekAtLastError() { return last; }

hipError_t hipStreamCreate(hipStream_t* s) {
  *s = reinterpret_cast<hipStream_t>(8);
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t* s, unsigned) { return hipStreamCreate(s); }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return sync(); }
hipError_t hipStreamQuery(hipStream_t) {
  if (broken) return ret(hipErrorLaunchFailure);
  std::lock_guard<std::mutex> lk(qmu);
  return queue.empty() ? hipSuccess : ret(hipErrorNotReady);
}
hipError_t hipEventCreate(hipEvent_t* e) {
  *e = reinterpret_cast<hipEvent_t>(8);
  return hipSuccess;
}
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
hipError_t hipEventElapsedTime(float* ms, hipEvent_t, hipEvent_t) {
  *ms = 0.f;
  return hipSuccess;
}

hipError_t hipStreamBeginCapture(hipStream_t, hipStreamCaptureMode) {
  capturing = new Graph;
  return hipSuccess;
}
hipError_t hipStreamEndCapture(hipStream_t, hipGraph_t* g) {
  *g = reinterpret_cast<hipGraph_t>(capturing);
  capturing = nullptr;
  return hipSuccess;
}
hipError_t hipGraphGetNodes(hipGraph_t g, hipGraphNode_t*, size_t* n) {
  *n = reinterpret_cast<Graph*>(g)->nodes;
  return hipSuccess;
}
hipError_t hipGraphInstantiate(hipGraphExec_t* e, hipGraph_t g, hipGraphNode_t*, char*, size_t) {
  const Graph* q = reinterpret_cast<Graph*>(g);
  note("instantiate " + std::to_string(q->nodes));
  *e = reinterpret_cast<hipGraphExec_t>(new Graph(*q));
  return hipSuccess;
}
hipError_t hipGraphLaunch(hipGraphExec_t e, hipStream_t) {
  const Graph* q = reinterpret_cast<Graph*>(e);
  note("graph " + std::to_string(q->nodes));
  for (const Op& o : q->ops) submit(o);
  return hipSuccess;
}
hipError_t hipGraphDestroy(hipGraph_t g) {
  delete reinterpret_cast<Graph*>(g);
  return hipSuccess;
}
hipError_t hipGraphExecDestroy(hipGraphExec_t e) {
  delete reinterpret_cast<Graph*>(e);
  return hipSuccess;
}

}  // extern "C"
