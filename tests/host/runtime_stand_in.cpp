// A stand-in of the HIP runtime for host-only checks of the library (no GPU): device and pinned memory are plain host
// memory, streams and events do nothing, a kernel launch only counts and may be made to fail.  The library's objects are
// linked with it in place of the runtime.  The knobs and counters are declared in runtime_stand_in.hpp.
#include "runtime_stand_in.hpp"

#include <sys/mman.h>

#include <cstdint>
#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace stand_in {
size_t limit = ~size_t(0);
size_t live = 0, peak = 0;
long syncs = 0;
std::string fail_launch;
void* capturing = nullptr;
std::map<std::string, long> launches;
std::function<void(const std::string&, unsigned, void**)> on_launch;
static std::mutex mu;
static std::map<void*, size_t> sizes;
static std::map<const void*, std::string> names;
static int last_error = 0;

std::vector<std::string> kernels(const std::string& part) {
  std::vector<std::string> out;
  for (const auto& kv : names)
    if (kv.second.find(part) != std::string::npos) out.push_back(kv.second);
  return out;
}
long launched(const std::string& part) {
  long n = 0;
  for (const auto& kv : launches)
    if (kv.first.find(part) != std::string::npos) n += kv.second;
  return n;
}
}  // namespace stand_in

using namespace stand_in;

namespace {
constexpr int kOutOfMemory = 2, kLaunchFailure = 719, kCaptured = 907, kUnsupported = 900;
struct Dim3 {
  uint32_t x, y, z;
};
int set(int e) {
  if (e != 0) last_error = e;
  return e;
}
struct Config {
  Dim3 grid, block;
  size_t shared;
  void* stream;
};
thread_local Config config;
int new_handle(void** p) {
  *p = std::malloc(16);
  return 0;
}
}  // namespace

extern "C" {
int hipMalloc(void** p, size_t n) {
  std::lock_guard<std::mutex> lk(mu);
  *p = nullptr;
  if (live + n > limit) return set(kOutOfMemory);
  // address space alone until it is touched
  *p = mmap(nullptr, n, PROT_READ | PROT_WRITE, MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  if (*p == MAP_FAILED) {
    *p = nullptr;
    return set(kOutOfMemory);
  }
  sizes[*p] = n;
  live += n;
  if (live > peak) peak = live;
  return 0;
}
int hipFree(void* p) {
  std::lock_guard<std::mutex> lk(mu);
  if (!p) return 0;
  const auto it = sizes.find(p);
  if (it == sizes.end()) std::abort();  // not from hipMalloc, or freed before
  live -= it->second;
  munmap(p, it->second);
  sizes.erase(it);
  return 0;
}
int hipHostMalloc(void** p, size_t n, unsigned) {
  *p = std::malloc(n);
  return 0;
}
int hipHostFree(void* p) {
  std::free(p);
  return 0;
}
int hipHostGetDevicePointer(void** d, void* h, unsigned) {
  *d = h;
  return 0;
}
int hipMemcpy(void* d, const void* s, size_t n, int) {
  std::memcpy(d, s, n);
  return 0;
}
int hipMemcpyAsync(void* d, const void* s, size_t n, int, void*) {
  std::memcpy(d, s, n);
  return 0;
}
int hipMemsetAsync(void* d, int v, size_t n, void*) {
  std::memset(d, v, n);
  return 0;
}
int hipMemGetInfo(size_t* free_, size_t* total) {
  *free_ = limit - live;
  *total = limit;
  return 0;
}
int hipGetDeviceCount(int* n) {
  *n = 1;
  return 0;
}
int hipGetDevice(int* d) {
  *d = 0;
  return 0;
}
int hipSetDevice(int) { return 0; }
const char* hipGetErrorString(int e) { return e == kOutOfMemory ? "out of memory" : "error"; }
int hipGetLastError() {
  const int e = last_error;
  last_error = 0;
  return e;
}
int hipGetSymbolAddress(void** p, const void*) {
  *p = nullptr;
  return 0;
}
int hipStreamCreateWithFlags(void** s, unsigned) { return new_handle(s); }
int hipStreamDestroy(void* s) {
  std::free(s);
  return 0;
}
int hipStreamSynchronize(void* s) {
  ++syncs;
  return (capturing && s == capturing) ? kUnsupported : 0;
}
int hipStreamWaitEvent(void*, void*, unsigned) { return 0; }
int hipStreamIsCapturing(void* s, int* status) {
  *status = (capturing && s == capturing) ? 1 : 0;
  return 0;
}
int hipStreamBeginCapture(void*, int) { return 0; }
int hipStreamEndCapture(void*, void** g) { return new_handle(g); }
int hipGraphInstantiate(void** e, void*, void**, char*, size_t) { return new_handle(e); }
int hipGraphLaunch(void*, void*) { return 0; }
int hipGraphDestroy(void* g) {
  std::free(g);
  return 0;
}
int hipGraphExecDestroy(void* e) {
  std::free(e);
  return 0;
}
int hipEventCreate(void** e) { return new_handle(e); }
int hipEventCreateWithFlags(void** e, unsigned) { return new_handle(e); }
int hipEventDestroy(void* e) {
  std::free(e);
  return 0;
}
int hipEventRecord(void*, void*) { return 0; }
int hipEventQuery(void*) { return 0; }
int hipEventSynchronize(void*) { return capturing ? kCaptured : 0; }
int hipEventElapsedTime(float* ms, void*, void*) {
  *ms = 0.0f;
  return 0;
}
int hipLaunchKernel(const void* f, Dim3 grid, Dim3, void** args, size_t, void*) {
  std::lock_guard<std::mutex> lk(mu);
  const std::string& name = names[f];
  if (on_launch) on_launch(name, grid.y, args);
  if (!fail_launch.empty() && name.find(fail_launch) != std::string::npos) {
    fail_launch.clear();  // once
    return set(kLaunchFailure);
  }
  ++launches[name];
  return 0;
}
int __hipPushCallConfiguration(Dim3 g, Dim3 b, size_t sh, void* s) {
  config = Config{g, b, sh, s};
  return 0;
}
int __hipPopCallConfiguration(Dim3* g, Dim3* b, size_t* sh, void** s) {
  *g = config.grid;
  *b = config.block;
  *sh = config.shared;
  *s = config.stream;
  return 0;
}
void** __hipRegisterFatBinary(const void*) {
  static void* h;
  return &h;
}
void __hipUnregisterFatBinary(void**) {}
void __hipRegisterFunction(void**, const void* f, char*, const char* name, unsigned, void*, void*, void*, void*, int*) {
  std::lock_guard<std::mutex> lk(mu);
  names[f] = name;
}
void __hipRegisterVar(void**, void*, char*, const char*, int, size_t, int, int) {}
}
