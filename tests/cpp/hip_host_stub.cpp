// Stand-in for the HIP runtime, for tests of the library's host code without a
// GPU: device memory is host memory (lazily committed, zero), copies and fills
// are done, launches are recorded but not run, and a chosen call fails.  Loaded
// with RTLD_GLOBAL before libpbamd.so, it takes the place of the runtime's
// entry points that the library calls.
//
// Of the kernels only what the host code relies on is carried out: k_fill_u32,
// and the cell counters' life in a sort (the counting kernels leave them
// non-zero, k_scatter clears them).
#define __HIP_PLATFORM_AMD__ 1
#include <hip/hip_runtime_api.h>
#include <sys/mman.h>
#include <cstdint>
#include <cstring>
#include <map>
#include <string>
#include <vector>

namespace {
std::map<void *, size_t> live;                     // device allocations
std::map<const void *, std::string> kernels;       // host stub -> device name
std::map<const void *, void *> symbols;            // device variables
std::map<std::string, long> calls;
std::string fail_name;                             // call (or kernel) to fail, and which
long fail_at = 0;
hipError_t pending = hipSuccess;                   // what hipGetLastError will say
hipError_t launch_error = hipSuccess;
std::vector<std::string> launched;
uint64_t most_items = 0;                           // largest gridDim.x * blockDim.x
long dirty_counts = 0;
struct Config { dim3 g, b; size_t sh; hipStream_t st; };
std::vector<Config> configs;

hipError_t called(const char *name) {
  ++calls[name];
  if (fail_at > 0 && fail_name == name && --fail_at == 0) return hipErrorOutOfMemory;
  return hipSuccess;
}
void *take(size_t n) {
  void *p = mmap(nullptr, n ? n : 1, PROT_READ | PROT_WRITE,
                 MAP_PRIVATE | MAP_ANONYMOUS | MAP_NORESERVE, -1, 0);
  return p == MAP_FAILED ? nullptr : p;
}
template <typename T>
T arg(void **args, int k) { return *static_cast<T *>(args[k]); }
}  // namespace

extern "C" {
// ------------------------------------------------------------ test controls
void stub_fail(const char *name, long k) { fail_name = name; fail_at = k; }
void stub_pending_error() { pending = hipErrorInvalidValue; }
long stub_calls(const char *name) { return calls[name]; }
long stub_live() { return (long)live.size(); }
uint64_t stub_live_bytes() { uint64_t t = 0; for (auto &x : live) t += x.second; return t; }
uint64_t stub_most_items() { return most_items; }
long stub_dirty_counts() { return dirty_counts; }
long stub_launches(const char *name) {
  long n = 0;
  for (auto &k : launched) n += k.find(name) != std::string::npos;
  return n;
}
void stub_reset() { calls.clear(); launched.clear(); most_items = 0; fail_at = 0; }

// ------------------------------------------------------------------ memory
hipError_t hipMalloc(void **p, size_t n) {
  if (hipError_t e = called("hipMalloc")) return e;
  *p = take(n);
  live[*p] = n;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  auto it = live.find(p);
  if (it == live.end()) return hipErrorInvalidValue;
  munmap(p, it->second ? it->second : 1);
  live.erase(it);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t n, unsigned) {
  if (hipError_t e = called("hipHostMalloc")) return e;
  *p = take(n);
  return hipSuccess;
}
hipError_t hipHostFree(void *) { return hipSuccess; }
hipError_t hipHostGetDevicePointer(void **d, void *h, unsigned) { *d = h; return hipSuccess; }
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  if (hipError_t e = called("hipMemcpyAsync")) return e;
  std::memcpy(d, s, n);
  return hipSuccess;
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  if (v) std::memset(d, v, n);
  else if (n > (1u << 22)) madvise((void *)(((uintptr_t)d + 4095) & ~4095ull), (n - 4096) & ~4095ull, MADV_DONTNEED);
  else std::memset(d, 0, n);
  return hipSuccess;
}
hipError_t hipGetSymbolAddress(void **p, const void *sym) {
  *p = symbols[sym];
  return *p ? hipSuccess : hipErrorInvalidValue;
}

// ------------------------------------------------- devices, streams, events
hipError_t hipGetDeviceCount(int *n) { *n = 1; return hipSuccess; }
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof(*p));
  p->multiProcessorCount = 256;
  p->maxThreadsPerBlock = 1024;
  std::strcpy(p->gcnArchName, "host");
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) { *s = (hipStream_t)1; return hipSuccess; }
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return hipSuccess; }
hipError_t hipEventCreate(hipEvent_t *e) { *e = (hipEvent_t)1; return called("hipEventCreate"); }
hipError_t hipEventCreateWithFlags(hipEvent_t *e, unsigned) { return hipEventCreate(e); }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }
const char *hipGetErrorString(hipError_t) { return "stub error"; }
hipError_t hipGetLastError() {
  hipError_t e = pending ? pending : launch_error;
  pending = launch_error = hipSuccess;
  return e;
}

// ---------------------------------------------------------------- launches
void **__hipRegisterFatBinary(const void *) { static void *h; return &h; }
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *,
                           void *, void *, void *, int *) { kernels[host] = name; }
void __hipRegisterVar(void **, void *var, char *, char *, int, size_t n, int, int) { symbols[var] = take(n); }
hipError_t __hipPushCallConfiguration(dim3 g, dim3 b, size_t sh, hipStream_t st) {
  configs.push_back({g, b, sh, st});
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *g, dim3 *b, size_t *sh, hipStream_t *st) {
  const Config c = configs.back();
  configs.pop_back();
  *g = c.g; *b = c.b; *sh = c.sh; *st = c.st;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t, hipStream_t) {
  const std::string &name = kernels[f];
  const uint64_t items = (uint64_t)g.x * b.x;
  if (items > most_items) most_items = items;
  if (fail_at > 0 && name.find(fail_name) != std::string::npos && --fail_at == 0)
    return launch_error = hipErrorLaunchFailure;
  if (!items || items > 0xFFFFFFFFull) return launch_error = hipErrorInvalidConfiguration;
  launched.push_back(name);
  if (name.find("k_fill_u32") != std::string::npos) {
    uint32_t *x = arg<uint32_t *>(args, 0);
    for (uint32_t k = 0, n = arg<uint32_t>(args, 1); k < n; ++k) x[k] = arg<uint32_t>(args, 2);
  } else if (name.find("k_ref_bid") != std::string::npos || name.find("k_list_cellid") != std::string::npos) {
    uint32_t *counts = arg<uint32_t *>(args, 6);
    dirty_counts += counts[0] != 0;                // left by a sort that was given up
    ++counts[0];
  } else if (name.find("k_scatter") != std::string::npos) {
    std::memset(arg<uint32_t *>(args, 8), 0, 4 * (size_t)arg<uint32_t>(args, 9));
  }
  return hipSuccess;
}
hipError_t hipExtLaunchKernel(const void *f, dim3 g, dim3 b, void **args, size_t sh, hipStream_t st,
                              hipEvent_t, hipEvent_t, int) { return hipLaunchKernel(f, g, b, args, sh, st); }
}
