// Sits between libsvo and the HIP runtime in a child process (loaded before libsvo, with its symbols
// visible to it): every call goes on to the runtime, and where a trace launch keeps its tile costs is
// left for the test to read.
#include <dlfcn.h>
#include <hip/hip_runtime.h>

#include <cstring>
#include <set>

#include "svo_kernels.hpp"

namespace {

std::set<const void *> *g_trace;  // host addresses of the trace kernels
const uint32_t *g_cost;
uint32_t g_tiles, g_lanes;

template <class F>
F next(F, const char *name) {
  static void *hip = dlopen("libamdhip64.so.7", RTLD_NOW);
  return reinterpret_cast<F>(dlsym(hip, name));
}

}  // namespace

extern "C" {

const uint32_t *spy_cost() { return g_cost; }
uint32_t spy_tiles() { return g_tiles; }
uint32_t spy_lanes() { return g_lanes; }

void __hipRegisterFunction(void **modules, const void *host, char *device, const char *name, unsigned limit, void *tid,
                           void *bid, void *block, void *grid, int *size) {
  if (!g_trace) g_trace = new std::set<const void *>;
  if (std::strstr(name, "trace_frame_kernel")) g_trace->insert(host);
  next(&__hipRegisterFunction, "__hipRegisterFunction")(modules, host, device, name, limit, tid, bid, block, grid, size);
}

hipError_t hipLaunchKernel(const void *f, dim3 grid, dim3 block, void **args, size_t shared, hipStream_t s) {
  if (g_trace && g_trace->count(f)) {
    const auto &p = *static_cast<const svo::FrameParams *>(args[0]);
    g_cost = p.tile_cost;
    g_tiles = p.range_begin[8];
    g_lanes = p.lanes;
  }
  using Launch = hipError_t (*)(const void *, dim3, dim3, void **, size_t, hipStream_t);
  return next(Launch{}, "hipLaunchKernel")(f, grid, block, args, shared, s);
}

}  // extern "C"
