// Fused primary-frame cone tracer for gfx950 (MI355X).
//
// One persistent kernel replaces the reference's host-driven wavefront loop
// (MainWindow.RunWavefront/RunTraces, MainWindow.cs:356-481) and its kernels
// init / runBaseTrace / runBlockTrace / evaluateBackground / resolveRemainders /
// drawTrace (wavefront.cl:1352-1850).  Each lane owns one cone and runs the
// reference step machine to completion; because a cone's steps depend only on
// its own state and the read-only tree, the per-cone result equals the
// wavefront schedule's.
//
// MI355X mapping:
//   - persistent workgroups; idle lanes are refilled from a work counter with one
//     wave-aggregated atomic (ballot + popcount + mbcnt);
//   - 8 work ranges (bands of 8x8 pixel tiles), range r served first by the
//     workgroups of XCD r (blockIdx % 8), then stolen by the others, so each
//     XCD's L2 sees a spatially coherent part of the image;
//   - the dense Bases levels live in LDS; block records are fetched with one
//     128-bit load; instead of re-walking from the dense level every step
//     (getBlockAddress, wavefront.cl:296-304) each lane keeps a short stack of the
//     blocks it passed through in LDS ([level][lane]);
//   - the kernel is bound by VALU issue while the chip is full (a wave64 instruction is four
//     to five cycles of its SIMD) and by the instructions a lone wave issues (one in nine
//     cycles) while it waits for its longest cones, so the step loop has a form for ordinary
//     cones that does the same arithmetic in fewer instructions: masks, octants and pops from
//     the high words of the location, the minor axes' moves as two float-to-u32 conversions
//     without the saturation they cannot reach, the LOD tests through an approximate footprint
//     checked against its error, blocks without their addresses on the stack, usage ticks where
//     a block is entered instead of at every visit.  1080p depth-12 frame: 386.7 M -> 244.4 M
//     VALU instructions, 0.638 -> 0.484 ms a frame with three frames in flight, 0.87 -> 0.65 ms
//     alone; the 64-camera batch 8.34 -> 6.10 ms (VALU busy 99 %); forward + adjoint of 32 x 512^2
//     9.45 -> 6.75 ms (there the outputs of ended cones also moved out of the step loop).  Frames
//     that keep the general form gained from the rest: with depth of field 0.81 -> 0.72 ms alone,
//     with lanes refilled from 32 idle ones on 1.05 -> 0.90 ms;
//   - per-cone outputs are written by cone id; queue order is made canonical
//     (ascending cone id) by the order-preserving compaction kernels below.
#include <hip/hip_runtime.h>

#include <algorithm>
#include <type_traits>

#include "svo_device.hpp"
#include "svo_kernels.hpp"

namespace svo {

using namespace dev;

namespace {

__device__ __forceinline__ uint32_t lanes_below(uint64_t mask) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(mask >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)mask, 0u));
}

// WAVES > 0 asks the compiler for that many waves per SIMD (a register budget).
// HASH: the visit-sequence hash is computed only when its output is bound.
// Camera parameters come from the table p.cams (one camera or a batch), staged in LDS:
// kernel arguments stay small, so the scalar registers are not spilled.
// MODE: kModePlain ends a cone at its first material hit (the reference's frame);
// kModeComposite makes every hit a layer composited front to back and continues past the
// cell (up to p.max_layers layers); kModeAdjoint also back-propagates the L2 image loss to
// the layers' colour and opacity.
template <int WG, int WAVES, bool HASH, int MODE = kModePlain>
__global__ void __launch_bounds__(WG) __attribute__((amdgpu_waves_per_eu(WAVES > 0 ? WAVES : 1, 8)))
trace_frame_kernel(const FrameParams p) {
  extern __shared__ uint32_t smem[];
  uint16_t *s_bases = reinterpret_cast<uint16_t *>(smem);
  const uint32_t bases_words = p.bases_in_lds ? p.n_bases / 2u : 0u;
  uint32_t *s_cam = smem + bases_words;
  const uint32_t cam_words = p.n_cams * kCamWords;
  uint32_t *s_ticked = s_cam + cam_words;
  uint32_t *s_stack = s_ticked + p.ticked_slots;
  if (p.bases_in_lds) {
    // 16 bytes a load (Bases holds a multiple of 8 chunks and starts an allocation): chunk by chunk
    // the 18 dependent rounds of a BaseDepth-4 tree delayed every work-group's first cone
    const uint4 *src = reinterpret_cast<const uint4 *>(p.bases);
    uint4 *dst = reinterpret_cast<uint4 *>(s_bases);
    for (uint32_t i = threadIdx.x; i < p.n_bases / 8u; i += WG) dst[i] = src[i];
  }
  {
    const uint32_t *src = reinterpret_cast<const uint32_t *>(p.cams);
    for (uint32_t i = threadIdx.x; i < cam_words; i += WG) s_cam[i] = src[i];
  }
  for (uint32_t i = threadIdx.x; i < p.ticked_slots; i += WG) s_ticked[i] = kU32Max;
  __syncthreads();

  const uint32_t tid = threadIdx.x, lane = tid & 63u;
  const uint32_t B = p.B, S = p.stack_levels;
  const uint32_t xcd = blockIdx.x & 7u;
  // camera parameters: word w of camera c
  auto camf = [&](uint32_t c, uint32_t w) -> float { return __uint_as_float(s_cam[c * kCamWords + w]); };
  auto camu = [&](uint32_t c, uint32_t w) -> uint32_t { return s_cam[c * kCamWords + w]; };
  uint32_t cam = 0;    // the lane's camera
  float fov32 = 0.0f;  // fast steps: its cone FoV, scaled to distances in units of 2^-32
  // the frame tick travels with the camera records (word 21 of camera 0), so a captured
  // launch can be replayed for later frames
  const uint32_t tick = camu(0, 21);

  uint32_t range_step = 0;  // wave-uniform: ranges tried, in order xcd, xcd+1, ...
  bool fetching = true;     // wave-uniform
  uint32_t cur = 0, cur_end = 0, cur_t0 = 0;  // wave-uniform: the wave's claimed slice of work
  // the tile the wave took at its last refill (wave-uniform); its cost is the most steps any of
  // the lanes' cones took
  uint32_t cur_tile = kU32Max;

  bool active = false;
  uint32_t ray = 0, signs = 0, nvis = 0, nbase = 0;
  // The cone's level d is held as lv = 31 - d (level d's bit of a location is then bit lv of its
  // high word).  General steps go down to level 60: lv may be negative there.
  int lv = 31;
  // the location in sign-canonical form (c = x on an axis the cone moves down, ~x on one it
  // moves up: every axis then moves towards 0); loc(a) gives the location itself
  uint64_t cx = 0, cy = 0, cz = 0, hash = kFnvOffset;
  float dx = 0.f, dy = 0.f, dz = 0.f, ix = 0.f, iy = 0.f, iz = 0.f;
  uint32_t nchild = 0, nchunk = 0;  // Child field and chunk word of the current block
  // Morton code of the top min(depth, B) bits of the location: the level's Bases index is
  // powSum(depth - 1) + bm, kept up to date as the cone descends and pops instead of being
  // rebuilt from the location at every base step
  uint32_t bm = 0;
  float cone = 0.f;  // cone footprint at the current location, once cone_ok
  bool cone_ok = false;
  // 2^32 times the camera's coordinate measured along the canonical axis (fast steps); a stray cone
  // (below) has no use for them and keeps two block addresses in kx and ky
  float kx = 0.f, ky = 0.f, kz = 0.f;
  // A stray cone (not an ordinary one: a NaN, vanishing or huge direction) may move past cells
  // without crossing them level by level, so its block is the one it entered and not the one its
  // location names: it records the octant of each block it enters (bits 16..18 of the stacked
  // chunk word), the dense block's address (kx) and the current one's (ky).
  bool stray = false;
  uint32_t tot_vis = 0, tot_base = 0;
  // updateUsage is resolved one block late so its load never stalls the step.  A block's group is
  // ticked when a cone enters it: it is visited next.  Within a launch every write stores the same
  // frame tick, so a group needs its tick read (and, if it is not 65534/65535 and differs,
  // written) once: neither the deferral nor skipping a group already handled changes the result.
  // A group counts as handled when the workgroup's table of ticked groups (s_ticked,
  // direct-mapped) holds it; the lane that put it there writes it.
  uint32_t pend_g = kU32Max, pend_t = 0;
  auto resolve_usage = [&]() {
    if (pend_g != kU32Max && pend_t < 65534u && pend_t != (tick & 0xffffu))
      p.usage16[4u * (size_t)pend_g] = (uint16_t)tick;
    pend_g = kU32Max;
  };

  // The short stack holds, for each block level from B+2 down, the Child field and the chunk of
  // the block the cone passed through ([level][lane], one 64-bit word each), so a pop to a
  // stacked level needs no memory access.  The address of a block is its parent's Child field
  // plus its octant there, formed only when it is needed (block_address).
  uint2 *st_node = reinterpret_cast<uint2 *>(s_stack) + tid;
  const int lv_dense = 29 - (int)B;  // the dense block level B+2
  // Octant of the location at a level given by lv.
  auto octant = [&](int at, auto fast) -> uint32_t {
    if constexpr (decltype(fast)::value) {
      const uint32_t hx = (uint32_t)(cx >> 32), hy = (uint32_t)(cy >> 32), hz = (uint32_t)(cz >> 32);
      return (((hx >> at) & 1u) | (((hy >> at) & 1u) << 1) | (((hz >> at) & 1u) << 2)) ^ signs;
    } else {
      return chunk_position((uint32_t)(31 - at), cx, cy, cz) ^ signs;
    }
  };
  // Child field and chunk of the block of level `at` (a level the cone is still inside).
  auto stack_get = [&](int at) -> uint2 {
    const uint32_t rel = (uint32_t)(lv_dense - at), r = min(rel, S - 1u);
    uint2 q = st_node[r * WG];
    if (rel > r) {
      // deeper than the stack: walk down from its last level along the current location
      for (int l = lv_dense - (int)r; l > at; l--)
        q = load_node(p.blocks, p.n_blocks, q.x + (chunk_position((uint32_t)(31 - l), cx, cy, cz) ^ signs));
    }
    return q;
  };
  auto block_address = [&](int at) -> uint32_t {
    if (at >= lv_dense) {
      const uint32_t o0 = chunk_position(B, cx, cy, cz) ^ signs, o1 = chunk_position(B + 1u, cx, cy, cz) ^ signs;
      return (((bm << 3) | o0) << 3) | o1;
    }
    return stack_get(at + 1).x + (chunk_position((uint32_t)(30 - at), cx, cy, cz) ^ signs);
  };
  auto current_address = [&]() -> uint32_t { return stray ? __float_as_uint(ky) : block_address(lv); };
  // Returns to the block of level `at`: its Child field and chunk.
  auto pop_to = [&](int at, auto fast) {
    const uint2 q = stack_get(at);
    nchild = q.x;
    nchunk = q.y;
    if constexpr (!decltype(fast)::value) {
      if (stray) {
        const uint32_t rel = (uint32_t)(lv_dense - at);
        ky = rel == 0u ? kx
                       : __uint_as_float(rel < S ? st_node[(rel - 1u) * WG].x + ((q.y >> 16) & 7u) : block_address(at));
      }
    }
  };
  // Descends into the block at `addr` of level `at`, octant `oct` of its parent: fetches its Child
  // field and chunk (one 64-bit load), pushes them and ticks its usage group.
  auto enter = [&](int at, uint32_t addr, uint32_t oct, auto fast) {
    uint2 q = make_uint2(0u, 0u);
    if (addr < p.n_blocks) q = reinterpret_cast<const uint2 *>(p.blocks)[2u * (size_t)addr];
    const uint32_t g = addr >> 3;
    // (a cone at its step cap ends before it visits the block)
    if (g < p.n_usages && (decltype(fast)::value || nvis < kStepCap)) {
      const uint32_t slot = g & (p.ticked_slots - 1u);
      if (p.ticked_slots == 0u || s_ticked[slot] != g) {
        if (p.ticked_slots) s_ticked[slot] = g;
        resolve_usage();
        pend_g = g;
        pend_t = p.usage16[4u * (size_t)g];
      }
    }
    if constexpr (!decltype(fast)::value) {
      if (stray) {
        q.y = (q.y & 0xffffu) | (oct << 16);
        ky = __uint_as_float(addr);
        if (at == lv_dense) kx = ky;
      }
    }
    nchild = q.x;
    nchunk = q.y;
    const uint32_t rel = (uint32_t)(lv_dense - at);
    if (rel < S) st_node[rel * WG] = q;
  };

  // A cone that ends only records how (`fin`: bit0 pending, bit1 material, bit2 child request,
  // bit3 TreeSize, bit4 step cap, bit5 left the volume: an axis may stand one past its face);
  // its outputs are written when the wave next refills or exits, so the shading and output code
  // runs once for all lanes that ended in between instead of once per step in which any lane
  // ended.
  uint32_t fin = 0;
  auto retire = [&](uint32_t how) {
    fin = 1u | how;
    active = false;
  };
  // Writes the lane's ended cone: evaluateBackground / resolveRemainders / drawTrace for a primary
  // cone (weighting 255, parent = itself), plus the per-cone extension outputs.
  auto finish = [&]() {
    const bool material = fin & 2u, child = fin & 4u, tree_size = fin & 8u, capped = fin & 16u;
    uint32_t addr = kU32Max;
    float4 c;
    if (!material) {
      const float dp = (dx * 0.0f + dy * 0.0f) + dz * -1.0f;
      uint32_t r, g, b;
      if (dp > 0.8f) {
        r = g = b = 255u;
      } else {
        r = 135u;
        g = 206u;
        b = 235u;
      }
      const float fw = 255.0f * 255.0f;
      c = make_float4(fminf((float)(r * 255u) / fw, 1.0f), fminf((float)(g * 255u) / fw, 1.0f),
                      fminf((float)(b * 255u) / fw, 1.0f), 1.0f);
    } else {
      addr = current_address();
      if (addr == kU32Max) {
        c = make_float4(0.75f, 0.0f, 0.0f, 1.0f);
      } else {
        const uint4 q = load_block(p.blocks, p.n_blocks, addr);
        const float fw = 255.0f * 255.0f;
        c = make_float4(fminf((float)(block_r(q) * 255u) / fw, 1.0f), fminf((float)(block_g(q) * 255u) / fw, 1.0f),
                        fminf((float)(block_b(q) * 255u) / fw, 1.0f), 1.0f);
      }
    }
    const uint32_t depth = material ? (uint32_t)(31 - lv) : 0u;
    if (p.rgba) p.rgba[ray] = c;
    if (p.hit) p.hit[ray] = addr;
    if (p.visits) p.visits[ray] = nvis;
    if (HASH) p.hashes[ray] = hash;
    if (p.status) p.status[ray] = (uint8_t)((material ? 1u : 0u) | (child ? 2u : 0u) | (capped ? 4u : 0u));
    if (p.depth_out) p.depth_out[ray] = (uint8_t)depth;
    if (p.loc_out) {
      if (fin & 32u) {
        cx = cx == kU64Max ? 0ull : cx;
        cy = cy == kU64Max ? 0ull : cy;
        cz = cz == kU64Max ? 0ull : cz;
      }
      p.loc_out[4 * (size_t)ray + 0] = cx ^ sign_mask64(signs, 0u);
      p.loc_out[4 * (size_t)ray + 1] = cy ^ sign_mask64(signs, 1u);
      p.loc_out[4 * (size_t)ray + 2] = cz ^ sign_mask64(signs, 2u);
    }
    if (child && p.req_sparse) {
      svo_child_request rq;
      rq.address = addr;
      rq.tick = (uint16_t)tick;
      rq.depth = (uint8_t)depth;
      rq.pad0 = 0;
      rq.location[0] = cx ^ sign_mask64(signs, 0u);
      rq.location[1] = cy ^ sign_mask64(signs, 1u);
      rq.location[2] = cz ^ sign_mask64(signs, 2u);
      rq.tree_size = tree_size ? 1 : 0;
      for (int k = 0; k < 7; k++) rq.pad1[k] = 0;
      p.req_sparse[ray] = rq;
      if (p.req_keys) p.req_keys[ray] = make_uint2(addr, depth | (tree_size ? 256u : 0u));
    }
  };

  // ---- compositing state (composite modes) ----
  float cT = 1.0f, cR = 0.0f, cG = 0.0f, cB = 0.0f;  // transmittance, colour so far
  uint32_t nlay = 0, lay[kMaxLayers] = {kU32Max, kU32Max, kU32Max, kU32Max};  // indexed by constants only
  double loss_acc = 0.0;
  auto leaf = [&](uint32_t a) -> float4 {
    return a < p.n_blocks ? p.leaf_params[a] : make_float4(0.0f, 0.0f, 0.0f, 0.0f);
  };
  // one layer: C += T a c, T *= 1 - a
  auto composite = [&](uint32_t a) {
    const float4 q = leaf(a);
    const float w = cT * q.w;
    cR += w * q.x;
    cG += w * q.y;
    cB += w * q.z;
    cT = cT * (1.0f - q.w);
#pragma unroll
    for (uint32_t i = 0; i < kMaxLayers; i++) lay[i] = i == nlay ? a : lay[i];
    nlay++;
  };
  // The cone ended: the background takes the remaining transmittance; image, layers, loss
  // and (adjoint) the gradient of every layer.
  auto finish_composite = [&]() {
    const float dp = (dx * 0.0f + dy * 0.0f) + dz * -1.0f;
    const bool sun = dp > 0.8f;
    const float bg0 = sun ? 1.0f : 135.0f / 255.0f, bg1 = sun ? 1.0f : 206.0f / 255.0f,
                bg2 = sun ? 1.0f : 235.0f / 255.0f;
    const float C0 = cR + cT * bg0, C1 = cG + cT * bg1, C2 = cB + cT * bg2;
    if (p.rgba) p.rgba[ray] = make_float4(C0, C1, C2, 1.0f);
    if (p.layers_out)
#pragma unroll
      for (uint32_t i = 0; i < kMaxLayers; i++)
        if (i < p.max_layers) p.layers_out[(size_t)ray * p.max_layers + i] = i < nlay ? lay[i] : kU32Max;
    if (p.target) {
      const float4 t = p.target[ray];
      const float e0 = C0 - t.x, e1 = C1 - t.y, e2 = C2 - t.z;
      loss_acc += (double)e0 * e0 + (double)e1 * e1 + (double)e2 * e2;
      if (MODE == kModeAdjoint) {
        const float g0 = 2.0f * e0, g1 = 2.0f * e1, g2 = 2.0f * e2;
        // transmittance in front of each layer, then the composite behind it (back to front)
        float Ti[kMaxLayers];
        float T = 1.0f;
#pragma unroll
        for (uint32_t i = 0; i < kMaxLayers; i++) {
          Ti[i] = T;
          if (i < nlay) T = T * (1.0f - leaf(lay[i]).w);
        }
        float U0 = bg0, U1 = bg1, U2 = bg2;
#pragma unroll
        for (int i = (int)kMaxLayers - 1; i >= 0; i--) {
          if ((uint32_t)i >= nlay) continue;
          const uint32_t a = lay[i];
          const float4 q = leaf(a);
          if (a < p.n_blocks) {
            float *gr = reinterpret_cast<float *>(p.grads + a);
            const float w = Ti[i] * q.w;
            atomicAdd(gr + 0, g0 * w);
            atomicAdd(gr + 1, g1 * w);
            atomicAdd(gr + 2, g2 * w);
            atomicAdd(gr + 3, Ti[i] * ((g0 * (q.x - U0) + g1 * (q.y - U1)) + g2 * (q.z - U2)));
          }
          U0 = q.w * q.x + (1.0f - q.w) * U0;
          U1 = q.w * q.y + (1.0f - q.w) * U1;
          U2 = q.w * q.z + (1.0f - q.w) * U2;
        }
      }
    }
  };
  auto flush = [&]() {
    if (fin) {
      if (MODE == kModePlain)
        finish();
      else
        finish_composite();
      resolve_usage();
      tot_vis += nvis;
      tot_base += nbase;
      fin = 0;
    }
  };
  auto record_cost = [&]() {
    if (p.tile_cost && cur_tile != kU32Max) {
      uint32_t a = nvis;
      for (int off = 32; off > 0; off >>= 1) a = max(a, (uint32_t)__shfl_xor((int)a, off));
      if (lane == 0u) atomicMax(&p.tile_cost[cur_tile], a);  // several waves may run a part of it each
    }
    cur_tile = kU32Max;
    if (!active) nvis = 0;
  };

  bool pend_adv = false;  // the current step was visited and advances
  // One step's visit (runBaseTrace / runBlockTrace up to the octant test, wavefront.cl:1400-1429,
  // 1465-1505): counts the step and tests the octant.  True when it holds geometry (the step
  // decides), false when it is empty (the step advances).
  auto visit = [&](uint32_t &oct_out, auto fast) -> bool {
    uint32_t chunk;
    if (lv >= lv_dense + 2) {
      // powSum(d - 1) = 8 + 64 + ... + 8^(d-1): octal 1...10, i.e. bits 3, 6, ..., 3(d-1)
      const uint32_t d = (uint32_t)(31 - lv);
      const uint32_t index = (0x249248u & ((1u << (3u * d)) - 1u)) + bm;
      if (p.bases_in_lds) {
        chunk = s_bases[index];
      } else {
        // a 32-bit read of the chunk pair (Bases holds an even number of chunks), so that
        // the two paths stay an LDS read and a global read
        const uint32_t w = reinterpret_cast<const uint32_t *>(p.bases)[index >> 1];
        chunk = (w >> (16u * (index & 1u))) & 0xffffu;
      }
      nbase++;
      if (HASH) hash = (hash ^ (((uint64_t)d << 32) | index)) * kFnvPrime;
    } else {
      chunk = nchunk;
      if (HASH) hash = (hash ^ (((uint64_t)(uint32_t)(31 - lv) << 32) | current_address())) * kFnvPrime;
    }
    const uint32_t o = octant(lv, fast);
    nvis++;
    oct_out = o;
    return ((chunk >> (2u * o)) & 2u) != 0u;
  };
  // True (and the cone ends) when the cone has reached the step cap (general steps only: fast
  // steps stop short of it).
  auto at_cap = [&]() -> bool {
    if (nvis < kStepCap) return false;
    retire(16u);
    return true;
  };

  // A loop iteration takes at most one advancing step and then one deciding step: a lane whose
  // step advances visits its next step at once (the block it needs is in registers or on
  // the short stack, never behind a load) and, when that step decides, takes it in the same
  // iteration; a step visited as advancing waits as pend_adv for the next iteration.  Lanes
  // then run the long advance and the decision together instead of in alternate iterations.
  //
  // fast: the iteration's cones are ordinary ones (see fast_cone below): levels 1..30, the high
  // words decide octants, masks and pops; no step cap; the minor axes' moves cannot saturate;
  // the footprint is compared through an approximation that is checked to be far enough from
  // every threshold.  The general form holds for every cone.
  auto iteration = [&](auto fast) {
    constexpr bool FAST = decltype(fast)::value;
    bool adv = pend_adv, dec = false;
    uint32_t oct = 0;
    pend_adv = false;
    if (!adv) {
      if (FAST || !at_cap()) {
        dec = visit(oct, fast);
        adv = !dec;
      }
    }
    if (adv) {
      // advance to the next cell boundary, pop levels that were left
      const int l0 = lv;
      bool leave;
      int l1;
      if constexpr (FAST) {
        const uint32_t px = (uint32_t)(cx >> 32), py = (uint32_t)(cy >> 32), pz = (uint32_t)(cz >> 32);
        leave = traverse_fast((uint32_t)l0, cx, cy, cz, dx, dy, dz, ix, iy, iz, signs);
        // compare_canon on the high words: the levels crossed upwards from the cone's
        const uint32_t x = ((uint32_t)(cx >> 32) & ~px) | ((uint32_t)(cy >> 32) & ~py) | ((uint32_t)(cz >> 32) & ~pz);
        l1 = min(l0 + (int)__builtin_ctz(~(x >> l0)), 30);
      } else {
        const uint32_t dd = (uint32_t)(31 - l0);
        const uint64_t px = cx, py = cy, pz = cz;
        traverse_canon(dd, cx, cy, cz, dx, dy, dz, ix, iy, iz, signs);
        leave = leaving_canon(cx, cy, cz);
        l1 = 31 - (int)compare_canon(dd, px, py, pz, cx, cy, cz);
      }
      cone_ok = false;
      if (leave) {
        retire(32u);
      } else {
        // a block level pops to the level it names, except that level B+1 (no blocks)
        // means the base level B; a pop to a shallower block level re-reads the stack
        if (l1 <= lv_dense) {
          if (l1 > l0) pop_to(l1, fast);
        } else {
          // a pop to a base level keeps the top nd bits: drop the Morton triples below them.
          // The level is never less than 1, so at level 1 the top bit itself may have
          // changed (the cone crossed the volume's middle plane): rebuild it from the location.
          l1 = max(l1, lv_dense + 2);
          bm >>= 3u * (uint32_t)(l1 - max(l0, lv_dense + 2));
          if (l1 == 30) bm = chunk_position(0u, cx, cy, cz) ^ signs;
        }
        lv = l1;
        // the next step: visited now; an advancing one waits for the next iteration
        if (FAST || !at_cap()) {
          dec = visit(oct, fast);
          pend_adv = !dec;
        }
      }
    }
    if (dec) {
      if (lv > lv_dense) {
        // runBaseTrace's descent, wavefront.cl:1400-1463
        if (lv > lv_dense + 2) {
          lv--;
          bm = (bm << 3) | oct;
        } else {
          // the dense level B+2: Morton code of the top B+2 bits (bm holds the top B)
          lv = lv_dense;
          const uint32_t below = octant(lv_dense + 1, fast);
          enter(lv, (((bm << 3) | oct) << 3) | below, below, fast);
        }
      } else {
        // geometry in this octant: cone-footprint LOD decision, wavefront.cl:1516-1538;
        // the footprint depends on the location only, so it is computed once per location
        if (!cone_ok) {
          bool exact = true;
          if constexpr (FAST) {
            const float ax = (float)(uint32_t)(cx >> 32) - kx, ay = (float)(uint32_t)(cy >> 32) - ky,
                        az = (float)(uint32_t)(cz >> 32) - kz;
            const float m = __builtin_amdgcn_sqrtf(__builtin_fmaf(az, az, __builtin_fmaf(ay, ay, ax * ax)));
            cone = m * fov32;
            exact = cone_unsure(m, cone);
          }
          if (exact)
            cone = cone_at(camf(cam, 9), camf(cam, 10), camf(cam, 11), cx ^ sign_mask64(signs, 0u),
                           cy ^ sign_mask64(signs, 1u), cz ^ sign_mask64(signs, 2u), camf(cam, 12),
                           camf(cam, 13), camf(cam, 14));
          cone_ok = true;
        }
        // the LOD rule's five outcomes: up to level B+2 and hit, up one level, request a
        // child (hit), down to the child, hit; with d = 31 - lv: cone > 2^-d, cone <> 2^-(d+1)
        const float edge = FAST ? __uint_as_float(((uint32_t)lv << 23) + (96u << 23)) : exp2_neg((uint32_t)(31 - lv));
        const float half = FAST ? __uint_as_float(((uint32_t)lv << 23) + (95u << 23)) : exp2_neg((uint32_t)(32 - lv));
        const bool up_top = cone > exp2_neg(B + 2u);
        const bool up_one = !up_top && cone > edge;
        const bool stay = !up_top && !up_one;
        const bool no_child = nchild == kU32Max;
        if (stay && !no_child && cone < half && lv >= 31 - (int)kMaxDepth + 1) {
          lv--;
          enter(lv, nchild + oct, oct, fast);
        } else if (up_one) {
          lv++;
          pop_to(lv, fast);
        } else {
          // requestChild, wavefront.cl:362-375; TreeSize = min(1, (uchar)ConeDepth - Depth)
          const bool child = stay && no_child;
          if (up_top) {
            lv = lv_dense;
            if (MODE != kModePlain || !FAST) pop_to(lv, fast);
          }
          const uint32_t how = 2u | (child ? 4u : 0u) | (child && cone <= half ? 8u : 0u);
          if (MODE == kModePlain) {
            retire(how);
          } else {
            composite(current_address());
            if (nlay >= p.max_layers)
              retire(2u);
            else
              pend_adv = true;  // a composited layer: the cone continues past the cell
          }
        }
      }
    }
  };

  for (;;) {
    // ---- refill idle lanes with new cones (wave-uniform control flow) ----
    const uint64_t idle = __ballot(!active && lane < p.lanes);
    const uint32_t n_idle = (uint32_t)__popcll(idle);
    bool fast_cone = false;  // the lane's cone may take fast steps
    if (fetching && (n_idle >= p.refill || n_idle == p.lanes)) {
      flush();
      record_cost();
      // claim a slice of `chunk` work items with one atomic when the wave's slice is used up
      while (cur >= cur_end && range_step < 8u) {
        const uint32_t r = (xcd + range_step) & 7u;
        const uint32_t limit = (p.range_begin[r + 1] - p.range_begin[r]) * 64u;
        uint32_t base = 0;
        if (lane == 0) base = atomicAdd(&p.counters[r * kCounterStride], p.chunk);
        base = __shfl(base, 0);
        if (base < limit) {
          cur = base;
          cur_end = min(base + p.chunk, limit);
          cur_t0 = p.range_begin[r];
        } else {
          range_step++;
        }
      }
      if (cur >= cur_end) {
        fetching = false;
      } else {
        const uint32_t k = cur + lanes_below(idle);
        const uint32_t take = min(n_idle, cur_end - cur);
        cur_tile = p.order ? p.order[cur_t0 + (cur >> 6)] : cur_t0 + (cur >> 6);
        cur += take;
        if (!active && lane < p.lanes && k < cur_end) {
          uint32_t tile = cur_t0 + (k >> 6);
          if (p.order) tile = p.order[tile];
          const uint32_t l = k & 63u;
          // the camera whose tiles hold this one: the last with tile_begin <= tile
          uint32_t lo = 0, hi = p.n_cams;
          while (hi - lo > 1u) {
            const uint32_t mid = (lo + hi) >> 1;
            if (camu(mid, 18) <= tile)
              lo = mid;
            else
              hi = mid;
          }
          cam = lo;
          tile -= camu(cam, 18);
          const uint32_t W = camu(cam, 15), H = camu(cam, 16), tiles_x = camu(cam, 17), ray0 = camu(cam, 19),
                         lut0 = camu(cam, 20);
          float f[9];
          for (int j = 0; j < 9; j++) f[j] = camf(cam, j);
          const uint32_t tx = tile % tiles_x, ty = tile / tiles_x;
          const uint32_t x = tx * 8u + (l & 7u), y = ty * 8u + (l >> 3);
          if (x < W && y < H) {
            // setupInitialTrace, wavefront.cl:563-595 (trig from the camera table)
            ray = ray0 + x + y * W;
            const float *lut = p.lut + lut0;
            const float cu = lut[x], su = lut[W + x];
            const float cv = lut[2u * W + y], sv = lut[2u * W + H + y];
            const float m0 = cu * cv, m1 = (0.0f - su) * cv, m2 = sv;
            dx = (f[0] * m0 + f[3] * m1) + f[6] * m2;
            dy = (f[1] * m0 + f[4] * m1) + f[7] * m2;
            dz = (f[2] * m0 + f[5] * m1) + f[8] * m2;
            ix = 1.0f / dx;
            iy = 1.0f / dy;
            iz = 1.0f / dz;
            signs = (dx >= 0.0f ? 1u : 0u) | (dy >= 0.0f ? 2u : 0u) | (dz >= 0.0f ? 4u : 0u);
            nvis = 0;
            nbase = 0;
            hash = kFnvOffset;
            cone_ok = false;
            pend_adv = false;
            if (MODE != kModePlain) {
              cT = 1.0f;
              cR = cG = cB = 0.0f;
              nlay = 0;
            }
            const float o[3] = {camf(cam, 9), camf(cam, 10), camf(cam, 11)};
            const float d[3] = {dx, dy, dz}, inv[3] = {ix, iy, iz};
            uint64_t ex, ey, ez;
            const bool entered = trace_into_volume(o, d, inv, camf(cam, 12), ex, ey, ez);
            if (!entered) ex = ey = ez = 0;
            cx = ex ^ sign_mask64(signs, 0u);
            cy = ey ^ sign_mask64(signs, 1u);
            cz = ez ^ sign_mask64(signs, 2u);
            bm = chunk_position(0u, ex, ey, ez);
            kx = canon_origin(o[0], signs & 1u);
            ky = canon_origin(o[1], signs & 2u);
            kz = canon_origin(o[2], signs & 4u);
            lv = 30;
            if (entered)
              active = true;
            else
              retire(0u);
            stray = !ordinary_directions(dx, dy, dz);
            fast_cone = !stray && cx != 0ull && cy != 0ull && cz != 0ull && ordinary_camera(o, camf(cam, 12), camf(cam, 13));
          }
        }
      }
    }
    if (__ballot(active) == 0ull) {
      if (!fetching) break;
      continue;
    }
    // All lanes were refilled together from one tile (its cones share a camera): fast steps
    // while every one of them is an ordinary cone.
    if (p.refill >= 64u && n_idle == p.lanes && __ballot(active && !fast_cone) == 0ull) {
      const int lead = __ffsll((unsigned long long)__ballot(active)) - 1;
      cam = (uint32_t)__builtin_amdgcn_readlane((int)cam, lead);
      fov32 = camf(cam, 12) * 2.3283064365386963e-10f;
      bool run = active;
      while (run) {
        iteration(std::true_type{});
        run = active && lv > 1 && nvis < kStepCap - 4u;
      }
    }
    // General steps until enough lanes are idle to refill: a lane leaves this loop when its cone
    // ends, so the exec mask keeps finished lanes' registers untouched.
    while (active) {
      iteration(std::false_type{});
      const uint32_t running = (uint32_t)__popcll(__ballot(active));
      if (fetching && 64u - running >= p.refill) break;
    }
  }

  flush();
  resolve_usage();  // a tick still pending (every cone ending resolves it; kept for safety)
  record_cost();

  // frame totals: one 64-bit atomic per wave
  uint32_t vb = tot_base, vk = tot_vis - tot_base;
  for (int off = 32; off > 0; off >>= 1) {
    vb += __shfl_xor(vb, off);
    vk += __shfl_xor(vk, off);
  }
  if (MODE != kModePlain && p.loss) {
    for (int off = 32; off > 0; off >>= 1) loss_acc += __shfl_xor(loss_acc, off);
    if (lane == 0) atomicAdd(p.loss, loss_acc);
  }
  if (lane == 0) {
    atomicAdd(&p.totals[0], (unsigned long long)vb);
    atomicAdd(&p.totals[1], (unsigned long long)vk);
  }
}

// ---- tile schedule ----

// Cost class of a tile: floor(log2(steps of its longest cone)) - 2, clamped to 0..kCostClasses-1 (tiles of
// fewer than 8 steps, and unmeasured ones, are class 0; 512 and more, class 7).
constexpr uint32_t kCostClasses = 8;
__device__ __forceinline__ uint32_t cost_class(uint32_t c) {
  const uint32_t l = c ? 31u - (uint32_t)__clz(c) : 0u;
  return l < 3u ? 0u : min(kCostClasses - 1u, l - 2u);
}

constexpr uint32_t kOrderThreads = 1024;

// One work-group per band: a stable counting sort of the band's tiles by cost class, most
// expensive class first, so that the tiles that ran longest in the previous frame start
// first and the frame does not end waiting on an expensive tile taken late.  Thread t
// owns a contiguous run of the band's tiles.
// With cls (LDS of at least (n + 1) / 2 bytes) the band's cost classes are staged there
// first, eight loads a thread in flight together, and both passes read them from LDS; without
// it each pass reads the costs from memory, one load per tile in turn (bands of 70K tiles, as
// in a 64-camera batch, took 140 us that way).
__device__ __forceinline__ void order_band(const uint32_t *cost, uint32_t *order, uint32_t b0, uint32_t n,
                                           uint8_t *cls) {
  __shared__ uint32_t s_wave[kCostClasses][kOrderThreads / 64];
  __shared__ uint32_t s_base[kCostClasses];
  // staged classes: two tiles a byte (tile i in the low nibble of byte i/2 when i is even),
  // each byte written whole by one thread
  const uint32_t n_bytes = (n + 1u) / 2u;
  if (cls) {
    for (uint32_t j0 = 0; j0 < n_bytes; j0 += 4u * kOrderThreads) {
      uint32_t c[8];
#pragma unroll
      for (uint32_t t = 0; t < 8u; t++) {
        const uint32_t i = 2u * (j0 + (t >> 1) * kOrderThreads + threadIdx.x) + (t & 1u);
        c[t] = i < n ? cost[b0 + i] : 0u;
      }
#pragma unroll
      for (uint32_t t = 0; t < 4u; t++) {
        const uint32_t byte = j0 + t * kOrderThreads + threadIdx.x;
        if (byte < n_bytes) cls[byte] = (uint8_t)(cost_class(c[2u * t]) | (cost_class(c[2u * t + 1u]) << 4));
      }
    }
    __syncthreads();
  }
  auto class_of = [&](uint32_t i) -> uint32_t {
    return cls ? ((uint32_t)cls[i >> 1] >> (4u * (i & 1u))) & 15u : cost_class(cost[b0 + i]);
  };
  const uint32_t per = (n + kOrderThreads - 1) / kOrderThreads;
  const uint32_t i0 = min(n, threadIdx.x * per), i1 = min(n, i0 + per);
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t cnt[kCostClasses];
#pragma unroll
  for (int c = 0; c < (int)kCostClasses; c++) cnt[c] = 0;
  for (uint32_t i = i0; i < i1; i++) {
    const uint32_t k = class_of(i);
#pragma unroll
    for (int c = 0; c < (int)kCostClasses; c++) cnt[c] += (k == (uint32_t)c) ? 1u : 0u;
  }
  // exclusive scan of each class count over the threads, in thread order
  uint32_t off[kCostClasses];
#pragma unroll
  for (int c = 0; c < (int)kCostClasses; c++) {
    uint32_t v = cnt[c];
    for (int d = 1; d < 64; d <<= 1) {
      const uint32_t t = __shfl_up(v, d);
      if (lane >= (uint32_t)d) v += t;
    }
    off[c] = v - cnt[c];
    if (lane == 63u) s_wave[c][wave] = v;
  }
  __syncthreads();
  if (threadIdx.x < kCostClasses) {
    const uint32_t c = threadIdx.x;
    uint32_t run = 0;
    for (uint32_t w = 0; w < kOrderThreads / 64; w++) {
      const uint32_t t = s_wave[c][w];
      s_wave[c][w] = run;
      run += t;
    }
    s_base[c] = run;  // the class total, for now
  }
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t run = 0;
    for (int c = (int)kCostClasses - 1; c >= 0; c--) {
      const uint32_t t = s_base[c];
      s_base[c] = run;
      run += t;
    }
  }
  __syncthreads();
#pragma unroll
  for (int c = 0; c < (int)kCostClasses; c++) off[c] += s_base[c] + s_wave[c][wave];
  for (uint32_t i = i0; i < i1; i++) {
    const uint32_t k = class_of(i);
    uint32_t pos = 0;
#pragma unroll
    for (int c = 0; c < (int)kCostClasses; c++) {
      if (k == (uint32_t)c) {
        pos = off[c];
        off[c]++;
      }
    }
    order[b0 + pos] = b0 + i;
  }
}

// True when every camera of the frame is within kViewMoved and kViewTurnCos of the view
// recorded in `saved` (a band's copy), which then takes the frame's views.  The band's threads
// share the cameras; the barrier inside __syncthreads_or orders every read of the copy
// before any write to it.
__device__ bool views_coherent(const CamRec *cams, uint32_t n, float *saved) {
  uint32_t far = 0;
  for (uint32_t c = threadIdx.x; c < n; c += blockDim.x) {
    const float *a = saved + (size_t)c * kViewWords;
    const CamRec &r = cams[c];
    float moved = 0.0f, dot = 0.0f, la = 0.0f, lb = 0.0f;
#pragma unroll
    for (int k = 0; k < 3; k++) {
      const float d = a[k] - r.origin[k];
      moved += d * d;
      dot += a[3 + k] * r.facing[k];
      la += a[3 + k] * a[3 + k];
      lb += r.facing[k] * r.facing[k];
    }
    const bool near = a[6] == 1.0f && moved < kViewMoved * kViewMoved && dot > kViewTurnCos * sqrtf(la * lb);
    far |= near ? 0u : 1u;
  }
  const bool coherent = __syncthreads_or((int)far) == 0;
  for (uint32_t c = threadIdx.x; c < n; c += blockDim.x) {
    float *a = saved + (size_t)c * kViewWords;
    const CamRec &r = cams[c];
#pragma unroll
    for (int k = 0; k < 3; k++) {
      a[k] = r.origin[k];
      a[3 + k] = r.facing[k];
    }
    a[6] = 1.0f;
    a[7] = 0.0f;
  }
  return coherent;
}

// The work a frame does before its trace launch, in one launch: work-group 0 clears the
// frame's counters and totals and writes the camera records that came in the kernel
// argument; work-group b < bands builds band b's tile order (cost order when the views
// are coherent with the band's recorded ones, raster order otherwise) and clears its costs.  The
// camera poses are read from the argument when they came inline (work-group 0 may still be
// writing the device records), from the device records otherwise (copied before this launch).
__global__ void __launch_bounds__(kOrderThreads) frame_begin_kernel(FrameBegin f) {
  if (blockIdx.x == 0) {
    const uint32_t i = threadIdx.x;
    if (i < 8u) f.counters[i * kCounterStride] = 0u;
    if (i < 4u) f.totals[i] = 0ull;
    if (i < f.n_cams * kCamWords)
      reinterpret_cast<uint32_t *>(f.cams)[i] = reinterpret_cast<const uint32_t *>(f.cam)[i];
  }
  extern __shared__ uint8_t s_cls[];
  if (blockIdx.x < f.bands) {
    const uint32_t b0 = f.range_begin[blockIdx.x], n = f.range_begin[blockIdx.x + 1] - b0;
    const CamRec *poses = f.n_cams ? f.cam : f.cams;
    if (views_coherent(poses, f.n_views, f.views + (size_t)blockIdx.x * f.n_views * kViewWords)) {
      order_band(f.cost, f.order, b0, n, f.stage ? s_cls : nullptr);
    } else {
      for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) f.order[b0 + i] = b0 + i;
    }
    __syncthreads();  // the order has read the costs, which the frame's waves raise from 0
    for (uint32_t i = threadIdx.x; i < n; i += blockDim.x) f.cost[b0 + i] = 0u;
  }
}

__global__ void zero_u32_kernel(uint32_t *p, uint32_t n) {
  for (uint32_t i = blockIdx.x * blockDim.x + threadIdx.x; i < n; i += gridDim.x * blockDim.x) p[i] = 0u;
}

// The device's floatToUlong / ulongToFloat (wavefront.cl:200-209) applied to an array, for
// comparing the device conversions with the host's over large samples.
__global__ void convert_kernel(uint32_t kind, const void *in, void *out, size_t n) {
  for (size_t i = (size_t)blockIdx.x * blockDim.x + threadIdx.x; i < n; i += (size_t)gridDim.x * blockDim.x) {
    if (kind == 0)
      static_cast<uint64_t *>(out)[i] = float_to_ulong(static_cast<const float *>(in)[i]);
    else
      static_cast<float *>(out)[i] = ulong_to_float(static_cast<const uint64_t *>(in)[i]);
  }
}

// ---- order-preserving status compaction (ascending cone id) ----

constexpr uint32_t kCompactThreads = 256;
constexpr uint32_t kCompactPerThread = 16;
constexpr uint32_t kCompactChunk = kCompactThreads * kCompactPerThread;

__device__ __forceinline__ void load_status16(const uint8_t *status, uint32_t n, uint32_t base, uint8_t s[16]) {
  if (base + 16u <= n) {
    const uint4 v = *reinterpret_cast<const uint4 *>(status + base);
    const uint32_t w[4] = {v.x, v.y, v.z, v.w};
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] = (uint8_t)(w[i >> 2] >> (8 * (i & 3)));
  } else {
#pragma unroll
    for (int i = 0; i < 16; i++) s[i] = (base + i < n) ? status[base + i] : 0xffu;
  }
}

// category bits of one status byte: bit0 background, bit1 material, bit2 child request
__device__ __forceinline__ uint32_t categories(uint8_t s) {
  if (s == 0xffu) return 0u;
  return ((s & 1u) ? 2u : 1u) | ((s & 2u) ? 4u : 0u);
}

// Exclusive scan of three counters over the 256 threads of a block.
__device__ void block_scan3(uint32_t v[3], uint32_t total[3]) {
  __shared__ uint32_t s_wave[3][kCompactThreads / 64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  uint32_t incl[3] = {v[0], v[1], v[2]};
#pragma unroll
  for (int c = 0; c < 3; c++)
    for (int off = 1; off < 64; off <<= 1) {
      const uint32_t t = __shfl_up(incl[c], off);
      if (lane >= (uint32_t)off) incl[c] += t;
    }
  if (lane == 63u)
    for (int c = 0; c < 3; c++) s_wave[c][wave] = incl[c];
  __syncthreads();
  for (int c = 0; c < 3; c++) {
    uint32_t before = 0, all = 0;
    for (uint32_t w = 0; w < kCompactThreads / 64; w++) {
      if (w < wave) before += s_wave[c][w];
      all += s_wave[c][w];
    }
    v[c] = before + incl[c] - v[c];
    total[c] = all;
  }
  __syncthreads();
}

__global__ void __launch_bounds__(kCompactThreads) status_count_kernel(const uint8_t *status, uint32_t n,
                                                                        uint32_t *counts) {
  const uint32_t base = blockIdx.x * kCompactChunk + threadIdx.x * kCompactPerThread;
  uint8_t s[16];
  load_status16(status, n, base, s);
  uint32_t v[3] = {0u, 0u, 0u};
#pragma unroll
  for (int i = 0; i < 16; i++) {
    const uint32_t c = categories(s[i]);
    v[0] += c & 1u;
    v[1] += (c >> 1) & 1u;
    v[2] += (c >> 2) & 1u;
  }
  uint32_t total[3];
  block_scan3(v, total);
  if (threadIdx.x == 0)
    for (int c = 0; c < 3; c++) counts[4u * blockIdx.x + c] = total[c];
}

// Single-workgroup exclusive scan of the per-chunk counts; writes the queue counters.  Thread
// t sums a contiguous run of chunks, one scan over the threads gives each run its start, and
// the thread writes its run's prefixes (one barrier round however many chunks).
__global__ void __launch_bounds__(kCompactThreads) status_scan_kernel(uint32_t *counts, uint32_t chunks,
                                                                       uint32_t *bg_count, uint32_t *mat_count,
                                                                       uint32_t *req_count,
                                                                       unsigned long long *totals) {
  uint4 *cnt = reinterpret_cast<uint4 *>(counts);
  const uint32_t per = (chunks + kCompactThreads - 1u) / kCompactThreads;
  const uint32_t c0 = min(chunks, threadIdx.x * per), c1 = min(chunks, c0 + per);
  uint32_t v[3] = {0u, 0u, 0u};
  for (uint32_t i = c0; i < c1; i++) {
    const uint4 t = cnt[i];
    v[0] += t.x;
    v[1] += t.y;
    v[2] += t.z;
  }
  uint32_t carry[3];
  block_scan3(v, carry);
  for (uint32_t i = c0; i < c1; i++) {
    const uint4 t = cnt[i];
    cnt[i] = make_uint4(v[0], v[1], v[2], t.w);
    v[0] += t.x;
    v[1] += t.y;
    v[2] += t.z;
  }
  if (threadIdx.x == 0) {
    if (bg_count) *bg_count = carry[0];
    if (mat_count) *mat_count = carry[1];
    if (req_count) *req_count = carry[2];
    totals[2] = carry[2];
  }
}

// Number of set bits of m below this lane.
__device__ __forceinline__ uint32_t rank_below(uint64_t m) {
  return __builtin_amdgcn_mbcnt_hi((uint32_t)(m >> 32), __builtin_amdgcn_mbcnt_lo((uint32_t)m, 0u));
}

// Wave w of a work-group writes the entries of cone ids [chunk + 1024 w, chunk + 1024 (w+1))
// in 16 rounds of 64 consecutive ids, one per lane: each round's entries of a queue go to
// consecutive positions (ranks from ballots), so the record reads and the queue writes are
// coalesced.  Positions continue the chunk offsets of the scan in ascending cone id.
// kFused (at most kFusedChunks chunks): `offsets` holds the chunks' own counts, each work-group
// sums those before it, and the last one writes the queue counters and the request total.
// kDirect (at most kDirectChunks chunks): there are no counts; each work-group counts the status
// bytes before its own.  One launch fewer: about 9 us of a small frame's 80 to 150, against at most
// 15 x 4096 bytes read again by the last work-group.
constexpr uint32_t kFusedChunks = 1024, kDirectChunks = 16;
enum : uint32_t { kScanned = 0, kFused = 1, kDirect = 2 };
__global__ void __launch_bounds__(kCompactThreads) status_scatter_kernel(
    const uint8_t *status, uint32_t n, const uint32_t *offsets, uint32_t *bg_queue, uint32_t *mat_queue,
    const svo_child_request *req_sparse, svo_child_request *requests, uint32_t *req_cones, uint32_t req_capacity,
    uint32_t mode, uint32_t *bg_count, uint32_t *mat_count, uint32_t *req_count, unsigned long long *totals) {
  uint32_t pre[3];
  if (mode == kDirect) {
    uint32_t v[3] = {0u, 0u, 0u};
    // (all of these bytes lie before this chunk, so none is past the end)
    for (uint32_t i = threadIdx.x * 16u; i < blockIdx.x * kCompactChunk; i += kCompactThreads * 16u) {
      uint8_t s[16];
      load_status16(status, n, i, s);
#pragma unroll
      for (int k = 0; k < 16; k++) {
        const uint32_t c = categories(s[k]);
        for (int q = 0; q < 3; q++) v[q] += (c >> q) & 1u;
      }
    }
    block_scan3(v, pre);
  } else if (mode == kFused) {
    uint32_t v[3] = {0u, 0u, 0u};
    for (uint32_t c = threadIdx.x; c < blockIdx.x; c += kCompactThreads)
      for (int q = 0; q < 3; q++) v[q] += offsets[4u * c + q];
    block_scan3(v, pre);
  } else {
    for (int q = 0; q < 3; q++) pre[q] = offsets[4u * blockIdx.x + q];
  }
  constexpr uint32_t kRounds = kCompactChunk / kCompactThreads;
  __shared__ uint32_t s_tot[3][kCompactThreads / 64];
  const uint32_t lane = threadIdx.x & 63u, wave = threadIdx.x >> 6;
  const uint32_t wbase = blockIdx.x * kCompactChunk + wave * (64u * kRounds);
  uint64_t cats = 0;  // 3 category bits per round
  uint32_t tot[3] = {0u, 0u, 0u};
#pragma unroll
  for (uint32_t r = 0; r < kRounds; r++) {
    const uint32_t id = wbase + r * 64u + lane;
    const uint32_t c = categories(id < n ? status[id] : (uint8_t)0xffu);
    cats |= (uint64_t)c << (3u * r);
#pragma unroll
    for (uint32_t q = 0; q < 3; q++) tot[q] += (uint32_t)__popcll(__ballot((c >> q) & 1u));
  }
  if (lane == 0)
    for (uint32_t q = 0; q < 3; q++) s_tot[q][wave] = tot[q];
  __syncthreads();
  uint32_t pos[3];
#pragma unroll
  for (uint32_t q = 0; q < 3; q++) {
    pos[q] = pre[q];
    for (uint32_t w = 0; w < wave; w++) pos[q] += s_tot[q][w];
  }
  if (mode != kScanned && blockIdx.x == gridDim.x - 1u && threadIdx.x == 0) {
    uint32_t all[3] = {pre[0], pre[1], pre[2]};
    for (uint32_t q = 0; q < 3; q++)
      for (uint32_t w = 0; w < kCompactThreads / 64; w++) all[q] += s_tot[q][w];
    if (bg_count) *bg_count = all[0];
    if (mat_count) *mat_count = all[1];
    if (req_count) *req_count = all[2];
    totals[2] = all[2];
  }
#pragma unroll
  for (uint32_t r = 0; r < kRounds; r++) {
    const uint32_t id = wbase + r * 64u + lane;
    const uint32_t c = (uint32_t)(cats >> (3u * r)) & 7u;
    const uint64_t m0 = __ballot(c & 1u), m1 = __ballot(c & 2u), m2 = __ballot(c & 4u);
    if ((c & 1u) && bg_queue) bg_queue[pos[0] + rank_below(m0)] = id;
    if ((c & 2u) && mat_queue) mat_queue[pos[1] + rank_below(m1)] = id;
    if (c & 4u) {
      const uint32_t at = pos[2] + rank_below(m2);
      if (requests && at < req_capacity) requests[at] = req_sparse[id];
      if (req_cones && at < req_capacity) req_cones[at] = id;
    }
    pos[0] += (uint32_t)__popcll(m0);
    pos[1] += (uint32_t)__popcll(m1);
    pos[2] += (uint32_t)__popcll(m2);
  }
}

template <int WG, int WAVES>
int launch_trace_wg(const FrameParams &p, const LaunchShape &shape, hipStream_t stream) {
  if (p.hashes)
    hipLaunchKernelGGL((trace_frame_kernel<WG, WAVES, true>), dim3(shape.grid), dim3(WG), shape.lds_bytes, stream, p);
  else
    hipLaunchKernelGGL((trace_frame_kernel<WG, WAVES, false>), dim3(shape.grid), dim3(WG), shape.lds_bytes, stream, p);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

// Occupancy of the hashing variant (never fewer registers than the plain one) bounds the
// grid of both.
template <int WG, int WAVES>
int occupancy_wg(size_t lds, int *blocks_per_cu) {
  return hipOccupancyMaxActiveBlocksPerMultiprocessor(blocks_per_cu, trace_frame_kernel<WG, WAVES, true>, WG, lds) ==
                 hipSuccess
             ? 0
             : -1;
}

template <int WAVES>
int launch_waves(const FrameParams &p, const LaunchShape &shape, hipStream_t stream) {
  switch (shape.workgroup) {
    case 64: return launch_trace_wg<64, WAVES>(p, shape, stream);
    case 128: return launch_trace_wg<128, WAVES>(p, shape, stream);
    case 256: return launch_trace_wg<256, WAVES>(p, shape, stream);
    case 512: return launch_trace_wg<512, WAVES>(p, shape, stream);
    case 1024: return launch_trace_wg<1024, WAVES>(p, shape, stream);
    default: return -1;
  }
}

template <int WAVES>
int occupancy_waves(int wg, size_t lds, int *blocks_per_cu) {
  switch (wg) {
    case 64: return occupancy_wg<64, WAVES>(lds, blocks_per_cu);
    case 128: return occupancy_wg<128, WAVES>(lds, blocks_per_cu);
    case 256: return occupancy_wg<256, WAVES>(lds, blocks_per_cu);
    case 512: return occupancy_wg<512, WAVES>(lds, blocks_per_cu);
    case 1024: return occupancy_wg<1024, WAVES>(lds, blocks_per_cu);
    default: return -1;
  }
}

}  // namespace

int trace_occupancy(int wg, int waves, size_t lds_bytes, int *blocks_per_cu) {
  switch (waves) {
    case 4: return occupancy_waves<4>(wg, lds_bytes, blocks_per_cu);
    case 5: return occupancy_waves<5>(wg, lds_bytes, blocks_per_cu);
    case 6: return occupancy_waves<6>(wg, lds_bytes, blocks_per_cu);
    default: return -1;
  }
}

int launch_frame_begin(const FrameBegin &f, hipStream_t stream) {
  if (f.n_cams > kInlineCams || f.bands > 8u) return -1;
  if (f.bands && (!f.views || !f.n_views || (f.n_cams && f.n_cams != f.n_views))) return -1;
  // bands of up to kStageTiles tiles stage their cost classes in LDS (two tiles a byte)
  constexpr uint32_t kStageTiles = 96u * 1024u;
  uint32_t most = 0;
  for (uint32_t b = 0; b < f.bands; b++) most = std::max(most, f.range_begin[b + 1] - f.range_begin[b]);
  FrameBegin g = f;
  g.stage = most > 0u && most <= kStageTiles ? 1u : 0u;
  const size_t lds = g.stage ? (size_t)(((most + 1u) / 2u + 15u) & ~15u) : 0;
  hipLaunchKernelGGL(frame_begin_kernel, dim3(std::max(1u, f.bands)), dim3(kOrderThreads), lds, stream, g);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_zero_u32(uint32_t *p, uint32_t n, hipStream_t stream) {
  if (n == 0) return 0;
  const uint32_t blocks = std::min<uint32_t>((n + 255u) / 256u, 1024u);
  hipLaunchKernelGGL(zero_u32_kernel, dim3(blocks), dim3(256), 0, stream, p, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_convert(uint32_t kind, const void *in, void *out, size_t n, hipStream_t stream) {
  if (n == 0) return 0;
  const uint32_t blocks = (uint32_t)std::min<size_t>((n + 255) / 256, 8192);
  hipLaunchKernelGGL(convert_kernel, dim3(blocks), dim3(256), 0, stream, kind, in, out, n);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

int launch_trace_frame(const FrameParams &p, const LaunchShape &shape, hipStream_t stream) {
  switch (shape.waves) {
    case 4: return launch_waves<4>(p, shape, stream);
    case 5: return launch_waves<5>(p, shape, stream);
    case 6: return launch_waves<6>(p, shape, stream);
    default: return -1;
  }
}

// The compositing modes hold more live state per lane (layers, colour, transmittance):
// they are compiled for 4 waves per SIMD.
int composite_occupancy(size_t lds_bytes, int *blocks_per_cu) {
  int a = 0, b = 0;
  if (hipOccupancyMaxActiveBlocksPerMultiprocessor(&a, trace_frame_kernel<256, 4, false, kModeComposite>, 256,
                                                   lds_bytes) != hipSuccess ||
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&b, trace_frame_kernel<256, 4, false, kModeAdjoint>, 256,
                                                   lds_bytes) != hipSuccess)
    return -1;
  *blocks_per_cu = a < b ? a : b;
  return 0;
}

int launch_composite(const FrameParams &p, const LaunchShape &shape, int mode, hipStream_t stream) {
  if (shape.workgroup != 256 || !p.n_cams) return -1;
  if (mode == kModeComposite)
    hipLaunchKernelGGL((trace_frame_kernel<256, 4, false, kModeComposite>), dim3(shape.grid), dim3(256),
                       shape.lds_bytes, stream, p);
  else if (mode == kModeAdjoint)
    hipLaunchKernelGGL((trace_frame_kernel<256, 4, false, kModeAdjoint>), dim3(shape.grid), dim3(256),
                       shape.lds_bytes, stream, p);
  else
    return -1;
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

uint32_t compaction_chunks(uint32_t n) { return (n + kCompactChunk - 1u) / kCompactChunk; }

int launch_compaction(const CompactParams &c, hipStream_t stream) {
  const uint32_t chunks = compaction_chunks(c.n);
  if (chunks == 0) return 0;
  if (chunks > kDirectChunks)
    hipLaunchKernelGGL(status_count_kernel, dim3(chunks), dim3(kCompactThreads), 0, stream, c.status, c.n, c.counts);
  if (chunks <= kFusedChunks) {
    hipLaunchKernelGGL(status_scatter_kernel, dim3(chunks), dim3(kCompactThreads), 0, stream, c.status, c.n, c.counts,
                       c.bg_queue, c.mat_queue, c.req_sparse, c.requests, c.req_cones, c.req_capacity,
                       chunks > kDirectChunks ? kFused : kDirect, c.bg_count, c.mat_count, c.req_count, c.totals);
    return hipGetLastError() == hipSuccess ? 0 : -1;
  }
  hipLaunchKernelGGL(status_scan_kernel, dim3(1), dim3(kCompactThreads), 0, stream, c.counts, chunks, c.bg_count,
                     c.mat_count, c.req_count, c.totals);
  hipLaunchKernelGGL(status_scatter_kernel, dim3(chunks), dim3(kCompactThreads), 0, stream, c.status, c.n, c.counts,
                     c.bg_queue, c.mat_queue, c.req_sparse, c.requests, c.req_cones, c.req_capacity, kScanned, c.bg_count,
                     c.mat_count, c.req_count, c.totals);
  return hipGetLastError() == hipSuccess ? 0 : -1;
}

}  // namespace svo
