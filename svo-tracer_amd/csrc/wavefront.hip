// Kernel-by-kernel wavefront path: HIP implementations of the reference kernels
// init / runBaseTrace / runBlockTrace / evaluateBackground / resolveRemainders /
// drawTrace (wavefront.cl:1352-1850) over the reference's per-ray SoA buffers,
// for callers that drive the frame loop from the host through svo_enqueue
// exactly as MainWindow.RunWavefront does (MainWindow.cs:356-622).
//
// Queue appends are deterministic and order-preserving (the reference's work-group atomic
// `increment`, wavefront.cl:249-287, leaves the order to the scheduler): a step's
// work-group of 1024 items counts its entries for each queue and either appends them
// itself (a step of one work-group) or leaves a code byte per item and its counts to
// append_kernel, whose work-groups sum the counts before their own.  A frame of the host
// loop is some 770 steps, most of a few thousand items at its end, so a step is bound by its
// launches: one or two instead of four, with coalesced appends (a thread that walked 16
// consecutive items took 12.9 us a launch), made the appends of the 1080p depth-12 loop
// 15.3 -> 1.7 ms of kernel time a frame and, with the counter read-backs below, the frame 28.4 ->
// 15.6 ms (the host calls included).
#include <hip/hip_runtime.h>

#include "svo_device.hpp"
#include "svo_wavefront_kernels.hpp"

namespace svo {

using namespace dev;

namespace {

constexpr uint32_t kThreads = 256;
constexpr uint32_t kStep = 1024;           // items of a step's work-group, one a thread

__device__ __forceinline__ void load_state(const WaveState &s, uint32_t id, float o[3], float d[3], float &fov,
                                           uint64_t &x, uint64_t &y, uint64_t &z, uint32_t &depth) {
  const float4 ov = s.origins[id], dv = s.directions[id];
  o[0] = ov.x;
  o[1] = ov.y;
  o[2] = ov.z;
  d[0] = dv.x;
  d[1] = dv.y;
  d[2] = dv.z;
  fov = s.fovs[id];
  x = s.locations[4 * (size_t)id + 0];
  y = s.locations[4 * (size_t)id + 1];
  z = s.locations[4 * (size_t)id + 2];
  depth = s.depths[id];
}

__device__ __forceinline__ void store_loc(const WaveState &s, uint32_t id, uint64_t x, uint64_t y, uint64_t z,
                                          uint32_t depth) {
  s.locations[4 * (size_t)id + 0] = x;
  s.locations[4 * (size_t)id + 1] = y;
  s.locations[4 * (size_t)id + 2] = z;
  s.depths[id] = (uint8_t)depth;
}

// getBlockAddress, wavefront.cl:296-304 (root-restart walk; the SoA state carries no stack).
__device__ __forceinline__ uint32_t walk_address(const uint4 *blocks, uint32_t n_blocks, uint32_t B, uint32_t depth,
                                                 uint64_t x, uint64_t y, uint64_t z) {
  uint32_t a = morton_top(B + 2u, x, y, z);
  for (uint32_t d = B + 2u; d < depth; d++) a = block_child(load_block(blocks, n_blocks, a)) + chunk_position(d, x, y, z);
  return a;
}

// init, wavefront.cl:1352-1398: the code of work-item (gx, gy); id is the cone it names.
__device__ __forceinline__ uint8_t init_item(const InitParams &p, uint32_t item, uint32_t &id) {
  const uint32_t gx = item % p.gsx, gy = item / p.gsx;
  id = gx + gy * p.W;
  if (id >= p.s.n_rays || gx >= p.W || gy >= p.H) return kCodeNone;
  const float cu = p.lut[gx], su = p.lut[p.W + gx], cv = p.lut[2u * p.W + gy], sv = p.lut[2u * p.W + p.H + gy];
  const float m0 = cu * cv, m1 = (0.0f - su) * cv, m2 = sv;
  float d[3], inv[3];
  for (int a = 0; a < 3; a++) {
    d[a] = (p.facing[a] * m0 + p.facing[3 + a] * m1) + p.facing[6 + a] * m2;
    inv[a] = 1.0f / d[a];
  }
  const float o[3] = {p.origin[0], p.origin[1], p.origin[2]};
  uint64_t lx = 0, ly = 0, lz = 0;
  const bool hit = trace_into_volume(o, d, inv, p.cone_fov, lx, ly, lz);
  if (hit) store_loc(p.s, id, lx, ly, lz, 1u);
  p.s.origins[id] = make_float4(o[0], o[1], o[2], 0.0f);
  p.s.directions[id] = make_float4(d[0], d[1], d[2], 0.0f);
  p.s.fovs[id] = p.cone_fov;
  p.s.parents[id] = id;
  p.s.weightings[id] = 255;
  if (p.colour_r) p.colour_r[id] = 0;
  if (p.colour_g) p.colour_g[id] = 0;
  if (p.colour_b) p.colour_b[id] = 0;
  p.final_r[id] = 0;
  p.final_g[id] = 0;
  p.final_b[id] = 0;
  p.final_w[id] = 0;
  return hit ? kQueueBase : kQueueBackground;
}

// runBaseTrace, wavefront.cl:1400-1463
__device__ __forceinline__ uint8_t base_item(const StepParams &p, uint32_t i, uint32_t &id) {
  uint8_t code = kCodeNone;
  id = p.in_queue[i];
  if (id < p.s.n_rays) {
    float o[3], d[3], fov;
    uint64_t x, y, z;
    uint32_t depth;
    load_state(p.s, id, o, d, fov, x, y, z, depth);
    const float ix = 1.0f / d[0], iy = 1.0f / d[1], iz = 1.0f / d[2];
    const uint32_t signs = (d[0] >= 0.0f ? 1u : 0u) | (d[1] >= 0.0f ? 2u : 0u) | (d[2] >= 0.0f ? 4u : 0u);
    const uint32_t B = p.B;
    if (depth >= 1u && depth <= B) {
      const uint32_t chunk = p.bases[base_offset(depth) + morton_top(depth, x, y, z)];
      if (((chunk >> (2u * chunk_position(depth, x, y, z))) & 2u) == 0u) {
        const uint64_t px = x, py = y, pz = z;
        traverse_chunk(depth, x, y, z, d[0], d[1], d[2], ix, iy, iz, signs);
        if (leaving(x, y, z, signs)) {
          depth = 0;
          code = kQueueBackground;
        } else {
          depth = compare_positions(depth, px, py, pz, x, y, z, signs);
          code = kQueueBase;
        }
      } else {
        depth = depth < B ? depth + 1u : B + 2u;
        if (depth == B + 1u) {
          depth = B;
          code = kQueueBase;
        } else {
          code = depth > B + 1u ? kQueueBlock : kQueueBase;
        }
      }
      store_loc(p.s, id, x, y, z, depth);
    }
  }
  return code;
}

// runBlockTrace, wavefront.cl:1465-1566
__device__ __forceinline__ uint8_t block_item(const StepParams &p, uint32_t i, uint32_t &id) {
  uint8_t code = kCodeNone;
  id = p.in_queue[i];
  if (id < p.s.n_rays) {
    float o[3], d[3], fov;
    uint64_t x, y, z;
    uint32_t depth;
    load_state(p.s, id, o, d, fov, x, y, z, depth);
    const uint32_t B = p.B;
    if (depth >= B + 2u && depth <= kMaxDepth) {
      const float ix = 1.0f / d[0], iy = 1.0f / d[1], iz = 1.0f / d[2];
      const uint32_t signs = (d[0] >= 0.0f ? 1u : 0u) | (d[1] >= 0.0f ? 2u : 0u) | (d[2] >= 0.0f ? 4u : 0u);
      const uint32_t addr = walk_address(p.blocks, p.n_blocks, B, depth, x, y, z);
      const uint4 blk = load_block(p.blocks, p.n_blocks, addr);
      const uint32_t g = addr >> 3;
      if (p.usage16 && g < p.n_usages) {
        const uint16_t t = p.usage16[4u * (size_t)g];
        if (t < 65534u && t != (uint16_t)p.tick) p.usage16[4u * (size_t)g] = (uint16_t)p.tick;
      }
      const float cone = cone_at(o[0], o[1], o[2], x, y, z, fov, p.dof0, p.dof1);
      const uint32_t oct = chunk_position(depth, x, y, z);
      bool complete = false, child = false;
      if (((block_chunk(blk) >> (2u * oct)) & 2u) == 0u) {
        const uint64_t px = x, py = y, pz = z;
        traverse_chunk(depth, x, y, z, d[0], d[1], d[2], ix, iy, iz, signs);
        if (leaving(x, y, z, signs)) {
          depth = 0;
          complete = true;
        } else {
          depth = compare_positions(depth, px, py, pz, x, y, z, signs);
        }
      } else if (cone > exp2_neg(B + 2u)) {
        depth = B + 2u;
        complete = true;
      } else if (cone > exp2_neg(depth)) {
        depth--;
      } else if (block_child(blk) == kU32Max) {
        child = true;
        complete = true;
      } else if (cone < exp2_neg(depth + 1u) && depth + 1u <= kMaxDepth) {
        depth++;
      } else {
        complete = true;
      }
      if (child && p.req_staging) {
        svo_child_request rq;
        rq.address = addr;
        rq.tick = (uint16_t)p.tick;
        rq.depth = (uint8_t)depth;
        rq.pad0 = 0;
        rq.location[0] = x;
        rq.location[1] = y;
        rq.location[2] = z;
        rq.tree_size = cone <= exp2_neg(depth + 1u) ? 1 : 0;
        for (int k = 0; k < 7; k++) rq.pad1[k] = 0;
        p.req_staging[i] = rq;
      }
      if (complete) {
        code = depth == 0 ? kQueueBackground : kQueueMaterial;
      } else {
        if (depth == B + 1u) depth = B;
        code = depth > B ? kQueueBlock : kQueueBase;
      }
      if (child) code |= kCodeRequest;
      store_loc(p.s, id, x, y, z, depth);
    }
  }
  return code;
}

// Whether an item with code c goes to target t (a queue, or the child requests).
__device__ __forceinline__ bool goes_to(uint8_t c, uint32_t t) {
  return t < 4u ? (c & 7u) == t : c != kCodeNone && (c & kCodeRequest) != 0u;
}

__device__ __forceinline__ uint32_t lanes_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Appends one wave's items (a lane each) behind pos[], which then counts them.
__device__ __forceinline__ void append_wave(const AppendParams &a, uint8_t c, uint32_t value, uint32_t staged,
                                            uint32_t pos[kAppendTargets]) {
#pragma unroll
  for (uint32_t t = 0; t < kAppendTargets; t++) {
    const bool in = goes_to(c, t);
    const uint64_t m = __ballot(in);
    const uint32_t at = pos[t] + lanes_below(m);
    if (in && at < a.capacity[t]) {
      if (t < 4u) {
        if (a.queue[t]) a.queue[t][at] = value;
      } else if (a.requests) {
        a.requests[at] = a.req_staging[staged];
      }
    }
    pos[t] += (uint32_t)__popcll(m);
  }
}

// One step (init, runBaseTrace or runBlockTrace) of 1024 work-items a work-group.  ONE: the step is
// one work-group, which appends its items and moves the counters itself.
enum { kInit, kBase, kBlock };
template <int KIND, bool ONE, class Params>
__global__ void __launch_bounds__(kStep) step_kernel(Params p, AppendParams a) {
  __shared__ uint32_t s_count[kAppendTargets][kStep / 64], s_from[kAppendTargets];
  const uint32_t i = blockIdx.x * kStep + threadIdx.x, lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint8_t code = kCodeNone;
  uint32_t id = 0;
  if (i < a.n) {
    if constexpr (KIND == kInit)
      code = init_item(p, i, id);
    else if constexpr (KIND == kBase)
      code = base_item(p, i, id);
    else
      code = block_item(p, i, id);
    if (!ONE) {
      a.codes[i] = code;
      a.values[i] = id;
    }
  }
#pragma unroll
  for (uint32_t t = 0; t < kAppendTargets; t++) {
    const uint32_t c = (uint32_t)__popcll(__ballot(goes_to(code, t)));
    if (lane == 0u) s_count[t][wave] = c;
  }
  // where the step's entries go: behind what each queue holds
  if (blockIdx.x == 0 && threadIdx.x < kAppendTargets)
    s_from[threadIdx.x] = a.counter[threadIdx.x] ? *a.counter[threadIdx.x] : 0u;
  __syncthreads();
  if (threadIdx.x < kAppendTargets) {
    const uint32_t t = threadIdx.x;
    uint32_t all = 0;
    for (uint32_t w = 0; w < kStep / 64u; w++) {
      const uint32_t c = s_count[t][w];
      if (ONE) s_count[t][w] = s_from[t] + all;
      all += c;
    }
    if (!ONE) {
      if (blockIdx.x == 0) a.from[t] = s_from[t];
      a.counts[kAppendTargets * blockIdx.x + t] = all;
    } else if (a.counter[t]) {
      *a.counter[t] = s_from[t] + all;
    }
  }
  if (ONE) {
    __syncthreads();
    uint32_t pos[kAppendTargets];
#pragma unroll
    for (uint32_t t = 0; t < kAppendTargets; t++) pos[t] = s_count[t][wave];
    append_wave(a, code, id, i, pos);
  }
}

// evaluateBackground, wavefront.cl:1741-1797 (the light mix of non-primary cones
// saturates its result to 0..255 where the reference's conversion is undefined)
__global__ void __launch_bounds__(kThreads) background_kernel(ShadeParams p) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= p.n) return;
  const uint32_t id = p.queue[i];
  if (id >= p.n_rays) return;
  const uint32_t parent = p.parents[id];
  if (parent >= p.n_pixels) return;
  const float4 dv = p.directions[id];
  const float dp = (dv.x * 0.0f + dv.y * 0.0f) + dv.z * -1.0f;
  uint32_t c[3];
  uint32_t lum;
  if (dp > 0.8f) {
    c[0] = c[1] = c[2] = 255u;
    lum = to_uchar(dp * 200.0f);
  } else {
    c[0] = 135u;
    c[1] = 206u;
    c[2] = 235u;
    lum = 1u;
  }
  const uint32_t w = p.weightings[id];
  if (w < 255u) {
    const uint32_t amb = p.ambient;
    const uint32_t boundary = lum > amb ? 255u : 0u;
    const uint32_t diff = lum > amb ? lum - amb : amb - lum;
    const float lq = (float)diff / ((float)(lum + amb) * 255.0f);
    const uint32_t base[3] = {p.colour_r ? p.colour_r[id] : 0u, p.colour_g ? p.colour_g[id] : 0u,
                              p.colour_b ? p.colour_b[id] : 0u};
    for (int k = 0; k < 3; k++) {
      const float v = (float)base[k] + lq * (float)c[k] * (float)(uint32_t)(boundary - base[k]);
      c[k] = to_uchar(v);
    }
  }
  atomicAdd(&p.final_w[parent], w);
  if (lum > 0u) {
    atomicAdd(&p.final_r[parent], c[0] * w);
    atomicAdd(&p.final_g[parent], c[1] * w);
    atomicAdd(&p.final_b[parent], c[2] * w);
  }
}

// resolveRemainders, wavefront.cl:1799-1833
__global__ void __launch_bounds__(kThreads) remainders_kernel(ShadeParams p) {
  const uint32_t i = blockIdx.x * kThreads + threadIdx.x;
  if (i >= p.n) return;
  const uint32_t id = p.queue[i];
  if (id >= p.n_rays) return;
  const uint32_t parent = p.parents[id];
  if (parent >= p.n_pixels) return;
  const uint32_t w = p.weightings[id];
  const uint64_t x = p.locations[4 * (size_t)id], y = p.locations[4 * (size_t)id + 1], z = p.locations[4 * (size_t)id + 2];
  const uint32_t depth = p.depths[id];
  if (depth < p.B + 2u || depth > kMaxDepth) return;
  const uint32_t a = walk_address(p.blocks, p.n_blocks, p.B, depth, x, y, z);
  if (a == kU32Max) return;
  const uint4 blk = load_block(p.blocks, p.n_blocks, a);
  atomicAdd(&p.final_w[parent], w);
  atomicAdd(&p.final_r[parent], block_r(blk) * w);
  atomicAdd(&p.final_g[parent], block_g(blk) * w);
  atomicAdd(&p.final_b[parent], block_b(blk) * w);
}

// drawTrace, wavefront.cl:1835-1850 (into a row-major float4 buffer instead of a GL image)
__global__ void __launch_bounds__(kThreads) draw_kernel(DrawParams p) {
  const uint32_t gx = blockIdx.x * kThreads + threadIdx.x, gy = blockIdx.y;
  if (gx >= p.gsx || gy >= p.gsy) return;
  const uint32_t id = gx + gy * p.W;
  if (id >= p.n_pixels || id >= p.n_out) return;
  const uint32_t w = p.final_w[id];
  float4 c;
  if (w == 0u) {
    c = make_float4(0.75f, 0.0f, 0.0f, 1.0f);
  } else {
    const float fw = (float)w * 255.0f;
    c = make_float4(fminf((float)p.final_r[id] / fw, 1.0f), fminf((float)p.final_g[id] / fw, 1.0f),
                    fminf((float)p.final_b[id] / fw, 1.0f), 1.0f);
  }
  p.out[id] = c;
}

// ---- order-preserving append of a step of several work-groups ----

// For steps of more than kSummed work-groups: exclusive sums of their counts, in place.  One
// work-group; thread t sums a run of them.
constexpr uint32_t kSummed = 4096;
__global__ void __launch_bounds__(kThreads) append_scan_kernel(uint32_t *counts, uint32_t steps) {
  __shared__ uint32_t s_run[kThreads];
  const uint32_t per = (steps + kThreads - 1u) / kThreads;
  const uint32_t b = min(steps, threadIdx.x * per), e = min(steps, b + per);
  for (uint32_t t = 0; t < kAppendTargets; t++) {
    uint32_t v = 0;
    for (uint32_t k = b; k < e; k++) v += counts[kAppendTargets * k + t];
    __syncthreads();
    s_run[threadIdx.x] = v;
    __syncthreads();
    uint32_t before = 0;
    for (uint32_t w = 0; w < threadIdx.x; w++) before += s_run[w];
    for (uint32_t k = b; k < e; k++) {
      const uint32_t c = counts[kAppendTargets * k + t];
      counts[kAppendTargets * k + t] = before;
      before += c;
    }
  }
}

// Work-group b appends the items of step work-group b: wave w its items 256w.., 64 consecutive ones a
// round, so queue and request writes are coalesced, with all four rounds' loads in flight together.
// summed: counts holds each step work-group's own counts, and those before b are summed here;
// otherwise their exclusive sums.  The last work-group moves the counters (which nothing else
// reads: a.from holds what they were).
__global__ void __launch_bounds__(kThreads) append_kernel(AppendParams a, uint32_t summed) {
  constexpr uint32_t kRounds = kStep / kThreads;
  __shared__ uint32_t s_before[kAppendTargets][kThreads / 64], s_own[kAppendTargets][kThreads / 64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6, first = blockIdx.x * kStep + wave * 64u * kRounds;
  uint8_t code[kRounds];
  uint32_t value[kRounds];
#pragma unroll
  for (uint32_t r = 0; r < kRounds; r++) {
    const uint32_t i = first + r * 64u + lane;
    code[r] = i < a.n ? a.codes[i] : kCodeNone;
    value[r] = i < a.n ? a.values[i] : 0u;
  }
  uint32_t before[kAppendTargets] = {0, 0, 0, 0, 0};
  if (summed) {
    for (uint32_t k = threadIdx.x; k < blockIdx.x; k += kThreads)
#pragma unroll
      for (uint32_t t = 0; t < kAppendTargets; t++) before[t] += a.counts[kAppendTargets * k + t];
#pragma unroll
    for (uint32_t t = 0; t < kAppendTargets; t++)
      for (int off = 32; off > 0; off >>= 1) before[t] += __shfl_xor(before[t], off);
  } else if (threadIdx.x == 0) {
#pragma unroll
    for (uint32_t t = 0; t < kAppendTargets; t++) before[t] = a.counts[kAppendTargets * blockIdx.x + t];
  }
#pragma unroll
  for (uint32_t t = 0; t < kAppendTargets; t++) {
    uint32_t own = 0;
#pragma unroll
    for (uint32_t r = 0; r < kRounds; r++) own += (uint32_t)__popcll(__ballot(goes_to(code[r], t)));
    if (lane == 0u) {
      s_before[t][wave] = before[t];
      s_own[t][wave] = own;
    }
  }
  __syncthreads();
  uint32_t pos[kAppendTargets];
#pragma unroll
  for (uint32_t t = 0; t < kAppendTargets; t++) {
    pos[t] = a.from[t];
    for (uint32_t w = 0; w < kThreads / 64u; w++) pos[t] += s_before[t][w] + (w < wave ? s_own[t][w] : 0u);
  }
#pragma unroll
  for (uint32_t r = 0; r < kRounds; r++) append_wave(a, code[r], value[r], first + r * 64u + lane, pos);
  if (blockIdx.x == gridDim.x - 1u && threadIdx.x == kThreads - 1u) {
#pragma unroll
    for (uint32_t t = 0; t < kAppendTargets; t++)
      if (a.counter[t]) *a.counter[t] = pos[t];
  }
}

// ResetIDBuffer's device half: the counter is cleared and goes to pinned host memory, tagged with the
// call's number.  The host returns on the word, without a wait for the stream, so the clear is
// released to the system before it: no work enqueued afterwards, on any stream, sees the old value.
__global__ void take_counter_kernel(uint32_t *counter, unsigned long long *host, uint32_t tag) {
  const uint32_t v = *counter;
  *counter = 0u;
  __hip_atomic_store(host, ((unsigned long long)tag << 32) | v, __ATOMIC_RELEASE, __HIP_MEMORY_SCOPE_SYSTEM);
}

template <int KIND, class Params>
int launch_step(const Params &p, const AppendParams &a, hipStream_t s) {
  if (a.n == 0u) return 0;
  const uint32_t steps = append_steps(a.n);
  if (steps == 1u) {
    hipLaunchKernelGGL((step_kernel<KIND, true, Params>), dim3(1), dim3(kStep), 0, s, p, a);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  hipLaunchKernelGGL((step_kernel<KIND, false, Params>), dim3(steps), dim3(kStep), 0, s, p, a);
  if (hipGetLastError() != hipSuccess) return -1;
  if (steps > kSummed) hipLaunchKernelGGL(append_scan_kernel, dim3(1), dim3(kThreads), 0, s, a.counts, steps);
  hipLaunchKernelGGL(append_kernel, dim3(steps), dim3(kThreads), 0, s, a, steps > kSummed ? 0u : 1u);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace

int launch_take_counter(uint32_t *counter, unsigned long long *host, uint32_t tag, hipStream_t s) {
  hipLaunchKernelGGL(take_counter_kernel, dim3(1), dim3(1), 0, s, counter, host, tag);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_init(const InitParams &p, const AppendParams &a, hipStream_t s) { return launch_step<kInit>(p, a, s); }

int launch_base_step(const StepParams &p, const AppendParams &a, hipStream_t s) { return launch_step<kBase>(p, a, s); }

int launch_block_step(const StepParams &p, const AppendParams &a, hipStream_t s) {
  return launch_step<kBlock>(p, a, s);
}

int launch_background(const ShadeParams &p, hipStream_t s) {
  hipLaunchKernelGGL(background_kernel, dim3((p.n + kThreads - 1) / kThreads), dim3(kThreads), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_remainders(const ShadeParams &p, hipStream_t s) {
  hipLaunchKernelGGL(remainders_kernel, dim3((p.n + kThreads - 1) / kThreads), dim3(kThreads), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_draw(const DrawParams &p, hipStream_t s) {
  hipLaunchKernelGGL(draw_kernel, dim3((p.gsx + kThreads - 1) / kThreads, p.gsy), dim3(kThreads), 0, s, p);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace svo
