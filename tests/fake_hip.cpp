// A HIP runtime without a device, for tests of the host code on the CPU.  Loaded before libsvo (with
// its symbols visible to it) it takes the place of libamdhip64: device memory is host memory of a
// bounded amount, a stream has finished whenever it is asked, and a kernel launch does nothing but
// leave its name and argument behind.  A call can be made to fail, and a failure stays the thread's
// last error until hipGetLastError, as it does in HIP since version 7.
#include <hip/hip_runtime.h>

#include <cstdlib>
#include <cstring>
#include <map>
#include <mutex>
#include <string>
#include <vector>

namespace {

std::mutex g_mutex;  // the calls come from several threads
using Lock = std::lock_guard<std::mutex>;
std::map<const void *, size_t> g_live;
size_t g_used = 0, g_limit = (size_t)4 << 30;
thread_local hipError_t g_last = hipSuccess;
std::string g_fail_call;
int g_fail_after = -1;
std::map<const void *, std::string> g_names;
std::vector<std::string> g_launches;
struct Config {
  dim3 grid, block;
  size_t shared;
  hipStream_t stream;
};
thread_local Config g_config;

hipError_t result(hipError_t e) {
  if (e != hipSuccess) g_last = e;
  return e;
}
// Whether this call is the one to fail.
bool fails(const char *call) { return g_fail_after >= 0 && g_fail_call == call && g_fail_after-- == 0; }
hipError_t step(const char *call) {
  Lock lock(g_mutex);
  return result(fails(call) ? hipErrorUnknown : hipSuccess);
}

}  // namespace

extern "C" {

// ---- what a test sets and asks ----
void fake_limit(size_t bytes) { g_limit = bytes; }
size_t fake_used() { return g_used; }
// The call after `after` more calls of this name fails, once.
void fake_fail(const char *call, int after) {
  g_fail_call = call;
  g_fail_after = after;
}
int fake_fail_pending() { return g_fail_after >= 0; }
size_t fake_launches() { return g_launches.size(); }

// ---- memory ----
hipError_t hipMalloc(void **p, size_t bytes) {
  Lock lock(g_mutex);
  *p = nullptr;
  if (fails("hipMalloc") || bytes > g_limit || g_used > g_limit - bytes) return result(hipErrorOutOfMemory);
  *p = std::calloc(1, bytes);
  if (!*p) return result(hipErrorOutOfMemory);
  g_live[*p] = bytes;
  g_used += bytes;
  return hipSuccess;
}
hipError_t hipFree(void *p) {
  Lock lock(g_mutex);
  auto it = g_live.find(p);
  if (it == g_live.end()) return result(hipErrorInvalidValue);
  g_used -= it->second;
  g_live.erase(it);
  std::free(p);
  return hipSuccess;
}
hipError_t hipHostMalloc(void **p, size_t bytes, unsigned) {
  *p = std::calloc(1, bytes);
  return step("hipHostMalloc");
}
hipError_t hipHostFree(void *p) {
  std::free(p);
  return hipSuccess;
}
hipError_t hipMemcpy(void *d, const void *s, size_t n, hipMemcpyKind) {
  std::memcpy(d, s, n);
  return step("hipMemcpy");
}
hipError_t hipMemcpyAsync(void *d, const void *s, size_t n, hipMemcpyKind, hipStream_t) {
  std::memcpy(d, s, n);
  return step("hipMemcpyAsync");
}
hipError_t hipMemsetAsync(void *d, int v, size_t n, hipStream_t) {
  std::memset(d, v, n);
  return step("hipMemsetAsync");
}

// ---- kernels ----
void **__hipRegisterFatBinary(const void *) {
  static void *handle;
  return &handle;
}
void __hipUnregisterFatBinary(void **) {}
void __hipRegisterFunction(void **, const void *host, char *, const char *name, unsigned, void *, void *, void *,
                           void *, int *) {
  g_names[host] = name;
}
void __hipRegisterVar(void **, void *, char *, char *, int, size_t, int, int) {}
hipError_t __hipPushCallConfiguration(dim3 grid, dim3 block, size_t shared, hipStream_t stream) {
  g_config = Config{grid, block, shared, stream};
  return hipSuccess;
}
hipError_t __hipPopCallConfiguration(dim3 *grid, dim3 *block, size_t *shared, hipStream_t *stream) {
  *grid = g_config.grid;
  *block = g_config.block;
  *shared = g_config.shared;
  *stream = g_config.stream;
  return hipSuccess;
}
hipError_t hipLaunchKernel(const void *f, dim3, dim3, void **, size_t, hipStream_t) {
  {
    Lock lock(g_mutex);
    g_launches.push_back(g_names[f]);
  }
  return step("hipLaunchKernel");
}
hipError_t hipOccupancyMaxActiveBlocksPerMultiprocessor(int *n, const void *, int block, size_t) {
  *n = 20 / (block / 64) > 0 ? 20 / (block / 64) : 1;
  return hipSuccess;
}

// ---- the rest ----
hipError_t hipGetLastError() {
  const hipError_t e = g_last;
  g_last = hipSuccess;
  return e;
}
const char *hipGetErrorString(hipError_t e) { return e == hipErrorOutOfMemory ? "out of memory" : "error"; }
hipError_t hipGetDeviceCount(int *n) {
  *n = 1;
  return hipSuccess;
}
hipError_t hipGetDevice(int *d) {
  *d = 0;
  return hipSuccess;
}
hipError_t hipSetDevice(int) { return hipSuccess; }
hipError_t hipGetDevicePropertiesR0600(hipDeviceProp_tR0600 *p, int) {
  std::memset(p, 0, sizeof *p);
  p->multiProcessorCount = 256;
  std::strcpy(p->gcnArchName, "gfx950");
  return hipSuccess;
}
hipError_t hipStreamCreateWithFlags(hipStream_t *s, unsigned) {
  *s = nullptr;
  return hipSuccess;
}
hipError_t hipStreamDestroy(hipStream_t) { return hipSuccess; }
hipError_t hipStreamSynchronize(hipStream_t) { return step("hipStreamSynchronize"); }
hipError_t hipStreamQuery(hipStream_t) { return hipSuccess; }
hipError_t hipDeviceSynchronize() { return step("hipDeviceSynchronize"); }
hipError_t hipEventCreate(hipEvent_t *) { return hipSuccess; }
hipError_t hipEventCreateWithFlags(hipEvent_t *, unsigned) { return hipSuccess; }
hipError_t hipEventDestroy(hipEvent_t) { return hipSuccess; }
hipError_t hipEventRecord(hipEvent_t, hipStream_t) { return hipSuccess; }
hipError_t hipEventSynchronize(hipEvent_t) { return hipSuccess; }

}  // extern "C"
