// k_wavefront.hip -- FP32 wavefront path tracer (radiance(), integrator.rs:53-135, split into
// kernels over SoA path queues).
//
// One pass renders `k` samples of a set of pixels: P = pixels * k paths, slot i -> pixel and
// sample by path_pixel (wavefront.h), so that neighbouring slots are samples of the same pixels.
// Per bounce:  extend (closest hit) -> shade (miss / RR / emission / NEE sampling / BSDF
// sampling; survivors compacted into the next queue) -> light self-occlusion -> shadow (any hit
// for the <= 2 NEE rays of each path, added to that path's radiance by the thread that owns the
// path).  The first bounce's extend and shade generate the camera rays themselves.
// After the last bounce, accumulate adds each pixel's k path radiances into FP64 sums.
// Queue compaction: a ballot per wave and one atomic per block on the block's queue segment.
// Random numbers: one PCG32 stream per (pixel, sample): seed_for(x, y, s) ^ seed.
#include "tpt_bsdf.h"
#include "tpt_kernels.h"
#include "tpt_sample32.h"
#include "tpt_selfocc64.h"
#include "tpt_trace32.h"
#include "wavefront.h"

#include <hip/hip_ext.h>

#include <algorithm>
#include <mutex>
#include <map>

namespace tpt {

// ---------------------------------------------------------------- queue compaction
// Position of this lane's entry in a queue when `pred` holds: a ballot per wave, the waves'
// counts combined in LDS, and one atomic per block, lanes ordered by block thread id.  Every
// thread of the block must call it (it synchronises the block); `sh` is 8 words of LDS.
__device__ __forceinline__ uint32_t block_slot(bool pred, uint32_t* __restrict__ count, uint32_t* sh) {
  const uint64_t mask = __ballot(pred);
  const uint32_t lane = __lane_id(), wave = threadIdx.x >> 6;
  if (lane == 0) sh[wave] = (uint32_t)__popcll(mask);
  __syncthreads();
  if (threadIdx.x == 0) {
    uint32_t tot = 0;
    for (uint32_t w = 0; w < TPT_WF_BLOCK / 64; w++) tot += sh[w];
    sh[7] = tot ? atomicAdd(count, tot) : 0u;
  }
  __syncthreads();
  uint32_t base = sh[7];
  for (uint32_t w = 0; w < wave; w++) base += sh[w];
  const uint32_t pos = base + (uint32_t)__popcll(mask & ((1ull << lane) - 1ull));
  __syncthreads();  // sh is reused by the next call
  return pos;
}

// Slot of this lane's entry in queue q (segment blockIdx % TPT_WF_SEGS) when `pred` holds, or
// UINT32_MAX (and the overflow flag raised) if the segment were full, which the segment size
// rules out.  Every thread of the block must call it.
__device__ __forceinline__ uint32_t seg_slot(bool pred, const PathState& ps, int q, uint32_t* sh) {
  const uint32_t g = blockIdx.x & (TPT_WF_SEGS - 1);
  const uint32_t pos = block_slot(pred, ps.counters + TPT_CNT_IDX(q, g), sh);
  if (pred && pos >= ps.seg_cap) {
    ps.counters[TPT_CNT_OVERFLOW] = 1u;
    return UINT32_MAX;
  }
  return g * ps.seg_cap + pos;
}

// ---------------------------------------------------------------- kernels
__device__ __forceinline__ uint32_t gtid() { return blockIdx.x * blockDim.x + threadIdx.x; }

// Path i of a pass (render.rs:142-157): its pixel and sample, its random stream
// seed_for(x, y, s) ^ seed, and its camera ray.  The first bounce's extension and shading
// kernels call it for their own paths, so no path state is written for bounce 0.
__device__ __forceinline__ void gen_path(const WfParams& W, const PassArgs& A, uint32_t i, RngF32* rng, f3* o, f3* d) {
  uint32_t pix, s;
  path_pixel(i, A.n_pixels, A.k, &pix, &s);
  if (A.active) {
    pix = (uint32_t)A.active[pix];
    s += A.nsamp[pix];
  } else {
    pix += A.pixel0;
    s += A.s0;
  }
  if (A.pix_map) pix = (uint32_t)A.pix_map[pix];
  const uint32_t x = pix % (uint32_t)W.width, y = pix / (uint32_t)W.width;
  *rng = RngF32(seed_for(x, y, s) ^ W.seed);
  camera_ray32(W.cam, x, y, W.inv_w, W.inv_h, *rng, o, d);
}

// Rays each wave takes at once: all 64 lanes while n rays fill the launched waves, else n spread
// over the waves (at least TPT_WF_MIN_LANES each).
__device__ __forceinline__ uint32_t lanes_per_wave(uint32_t n) {
  const uint32_t waves = gridDim.x * (TPT_WF_BLOCK / 64), q = (n + waves - 1) / waves;
  return max(min(q, 64u), (uint32_t)TPT_WF_MIN_LANES);
}

// A block's turns through the camera rays, a block's worth at a time: each round of gridDim.x pieces
// goes to the blocks in an order shifted against the last round's.  A fixed stride meets the same
// columns of the image whenever it is close to a multiple of its rows, and the blocks whose columns
// show the costly parts of the scene run on while the others are done: the first bounce's
// extension had 28% (Cornell box), 40% (1.31M-triangle mesh) and 31% (4096 instances) of the
// chip's wave slots filled where 62% can be.  Measured: Cornell 512^2 x 256 spp 21.57 -> 21.45 ms,
// the mesh at 1080p x 32 spp 33.5 -> 32.9, the instances adaptive 38.9 -> 37.8; shifting the shares of
// the later bounces' waves as well gave the instances 37.3 but took 1% from a 333 x 217 mesh render.
struct CameraTurns {
  uint32_t first, pos, step;
  __device__ __forceinline__ CameraTurns()
      : first(0), pos(blockIdx.x), step((uint32_t)((uint64_t)gridDim.x * 391 >> 10) | 1u) {}
  __device__ __forceinline__ bool any(uint32_t n) const { return first * TPT_WF_BLOCK < n; }
  __device__ __forceinline__ uint32_t ray() const { return (first + pos) * TPT_WF_BLOCK + threadIdx.x; }
  __device__ __forceinline__ void next() {
    first += gridDim.x;
    pos += step;
    if (pos >= gridDim.x) pos -= gridDim.x;
  }
};

// A pass without bounces (max_bounces 0) gathers no radiance: clear its paths' sums.
__global__ void __launch_bounds__(TPT_WF_BLOCK) k_clear_radiance(WfParams W, uint32_t n) {
  for (uint32_t i = gtid(); i < n; i += gridDim.x * blockDim.x) W.ps.L[i] = make_float4(0.f, 0.f, 0.f, 0.f);
}

__device__ __forceinline__ void tell_count(const WfParams& W, const PathCount& c) {
  if (gtid() != 0 || !c.seen) return;
  uint32_t n = 0;
  for (int g = 0; g < TPT_WF_SEGS; g++) n += W.ps.counters[TPT_CNT_IDX(c.queue ? TPT_CNT_Q1 : TPT_CNT_Q0, g)];
  __hip_atomic_store(c.seen, (uint64_t)c.tag << 32 | n, __ATOMIC_RELAXED, __HIP_MEMORY_SCOPE_SYSTEM);
}

// Every extension kernel: clears the queues that the shading kernel fills next, reports the paths,
// counts the n rays.
template <bool GEN>
__device__ __forceinline__ void begin_extension(const WfParams& W, int cur, uint32_t n, const PathCount& count) {
  if (gtid() < TPT_WF_SEGS) {
    W.ps.counters[TPT_CNT_IDX(cur ? TPT_CNT_Q0 : TPT_CNT_Q1, gtid())] = 0;
    W.ps.counters[TPT_CNT_IDX(TPT_CNT_SH, gtid())] = 0;
    W.ps.counters[TPT_CNT_IDX(TPT_CNT_SHL, gtid())] = 0;
    W.ps.counters[TPT_CNT_IDX(TPT_CNT_SHK, gtid())] = 0;
  }
  if (!GEN) tell_count(W, count);
  if (gtid() == 0) atomicAdd((unsigned long long*)&W.ps.stats[0], (unsigned long long)n);
}

// OVF: the scene's stack bound exceeds the LDS part, so the traversal stack may overflow to the
// per-thread global area (W.gstack); otherwise that path is compiled out.  GEN: the first
// bounce, whose paths are the pass's camera rays, generated here (path i at position i).  Six
// waves per SIMD fit the later bounces in 80 VGPRs without spills, five the first (its camera
// code needs more); the traversal is VALU-bound, and more waves hide its load latency.
template <bool OVF, bool GEN>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(GEN ? 5 : 6)))
k_extend(WfParams W, int cur, PassArgs A, PathCount count) {
  __shared__ int32_t s_stack[TPT_WF_STACK * TPT_WF_BLOCK];
  QueueMap qm;
  uint32_t n;
  if constexpr (GEN) {
    n = A.n_paths;
  } else {
    qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
    n = qm.n;
  }
  const float4* __restrict__ po = W.ps.o[cur];
  const float4* __restrict__ pd = W.ps.d[cur];
  LaneStackT<OVF> st{s_stack + threadIdx.x, OVF ? W.gstack + (size_t)gtid() * W.gstack_cap : nullptr, TPT_WF_BLOCK,
                     TPT_WF_STACK};
  begin_extension<GEN>(W, cur, n, count);
  auto trace = [&](uint32_t i, f3 o, f3 d) {
    HitF32 h;
    trace_f32<false>(W.S, o, d, (float)TPT_RAY_EPSILON, 1e30f, &h, st);
    W.ps.hit[i] = HitRec{__float_as_int(h.t), h.inst, h.prim};
  };
  if constexpr (GEN) {
    for (CameraTurns turn; turn.any(n); turn.next()) {
      const uint32_t i = turn.ray();
      if (i >= n) continue;
      f3 o, d;
      RngF32 rng(1);
      gen_path(W, A, i, &rng, &o, &d);
      trace(i, o, d);
    }
  } else {
    for (uint32_t i = gtid(); i < n; i += gridDim.x * blockDim.x) {
      const uint32_t slot = qm.slot(i);
      trace(i, f3of(po[slot]), f3of(pd[slot]));
    }
  }
}

// ---------------------------------------------------------------- small scenes (tpt_small32.h)
// A wave of k_extend_small / k_shadow_small starts rays once fewer lanes than this are tracing.
#define TPT_SMALL_LANES 25
#define TPT_SMALL_LANES_SH 17
// A wave's share of n entries, handed to its lanes as they fall idle: entry groups of 64, one
// group of every wave in turn, as a grid-stride loop takes them.  No atomics: the cursor is the
// wave's own.
struct WaveShare {
  uint32_t wave, waves, taken;
  __device__ __forceinline__ WaveShare()
      : wave((blockIdx.x * TPT_WF_BLOCK + threadIdx.x) >> 6), waves(gridDim.x * (TPT_WF_BLOCK / 64)), taken(0) {}
  // The next entry for this lane if it wants one; every lane of the wave must call it.
  __device__ __forceinline__ uint32_t take(bool want) {
    const uint64_t m = __ballot(want);
    const uint32_t c = taken + (uint32_t)__popcll(m & ((1ull << __lane_id()) - 1ull));
    taken += (uint32_t)__popcll(m);
    return ((c >> 6) * waves + wave) * 64 + (c & 63u);
  }
};

// The rays of a wave's share of queue cur, each lane's traversal resumable (TraceF32 step by step):
// once fewer than `lanes` lanes are tracing, the idle ones start their next rays, which they have
// held in registers since the last start, so that the wave does not wait for the load.
template <class Tree, class Stack>
__device__ __forceinline__ void extend_share(const WfParams& W, int cur, const Tree& tree, const Stack& st, int lanes) {
  QueueMap qm;
  qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
  const float4* __restrict__ po = W.ps.o[cur];
  const float4* __restrict__ pd = W.ps.d[cur];
  WaveShare share;
  TraceF32<false, Tree> tr;
  f3 no = mk(0.f, 0.f, 0.f), nd = no;
  uint32_t my = 0, nxt = 0;
  bool live = false, have = false;
  auto fetch = [&]() {  // every lane of the wave
    const uint32_t t = share.take(!have);
    if (have || t >= qm.n) return;
    nxt = t;
    have = true;
    const uint32_t slot = qm.slot(t);
    no = f3of(po[slot]);
    nd = f3of(pd[slot]);
  };
  fetch();
  for (;;) {
    const int nl = __popcll(__ballot(live));
    const bool some = __ballot(!live && have) != 0;
    if (some && nl < lanes) {  // wave-uniform
      if (!live && have) {
        my = nxt;
        have = false;
        live = tr.init(W.S, no, nd, (float)TPT_RAY_EPSILON, 1e30f);
        if (!live) W.ps.hit[my] = HitRec{__float_as_int(tr.hit.t), tr.hit.inst, tr.hit.prim};
      }
      fetch();
      continue;
    }
    if (nl == 0) break;  // the share is taken and every lane is idle
    if (live && !tr.step(W.S, st, tree)) {
      W.ps.hit[my] = HitRec{__float_as_int(tr.hit.t), tr.hit.inst, tr.hit.prim};
      live = false;
    }
  }
}

// k_extend for small scenes (SmallScene: at most 32 KB of trees, 20 stack entries, no instance
// but the flattened one).  k_extend spends its issue slots on idle lanes there -- 36% of the lanes of
// an instruction work on the Cornell box, since a wave ends with its longest ray -- and refilling
// waves from a global cursor stall on it, on the ray loads and, vector memory answering in order,
// then on their next node load.  Here the nodes and triangles are in LDS, whose loads are waited
// for apart from vector memory; a lane has its next ray in registers before it needs it (loaded
// while the wave traces); and a wave takes rays from its own share, without atomics.  Idle lanes
// start their rays once fewer than TPT_SMALL_LANES are tracing.  A ray's sequence of tests is
// k_extend's.  Cornell 512^2 x 256 spp 27.1 -> 22.3 ms (below 57 tracing lanes 23.5, 49 23.4, 33 and 17
// within 0.3% of 25, 9 1.5% slower); its adaptive render 28.6 -> 24.2; the inverse step's 16 spheres in
// the box and the sphere scene (bound by their short launches) unchanged.
// GEN: the first bounce's camera rays are coherent and need no loads, so a lane takes them as
// k_extend does.
template <bool GEN>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(GEN ? 5 : 6)))
k_extend_small(WfParams W, int cur, PassArgs A, PathCount count) {
  extern __shared__ float4 s_small[];
  QueueMap qm;
  uint32_t n;
  if constexpr (GEN) {
    n = A.n_paths;
  } else {
    qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
    n = qm.n;
  }
  LaneStackT<false> st;
  const SmallTree tree = load_small<TPT_WF_BLOCK>(W.S, W.small, s_small, &st);
  begin_extension<GEN>(W, cur, n, count);
  if constexpr (GEN) {
    for (CameraTurns turn; turn.any(n); turn.next()) {
      const uint32_t i = turn.ray();
      if (i >= n) continue;
      f3 o, d;
      RngF32 rng(1);
      gen_path(W, A, i, &rng, &o, &d);
      HitF32 h;
      trace_f32<false>(W.S, tree, o, d, (float)TPT_RAY_EPSILON, 1e30f, &h, st);
      W.ps.hit[i] = HitRec{__float_as_int(h.t), h.inst, h.prim};
    }
  } else {
    extend_share(W, cur, tree, st, TPT_SMALL_LANES);
  }
}

// Persistent form of k_extend for the later bounces of deep trees, where the rays of one wave need
// very different numbers of traversal steps: lanes that fall idle go on with the next rays of their
// wave's share once fewer than W.refill lanes are tracing (persistent threads, Aila and Laine 2009).
// The hits are those of k_extend: each ray's traversal is the same sequence of steps.  Against taking
// rays from one global cursor -- an atomic's and a ray load's way to memory, one after the other, for
// the whole wave at every start -- on MI355X: 1.31M-triangle mesh 1080p x 32 spp 36.7 -> 33.3 ms, 4096
// instances adaptive 46.7 -> 38.9, 20k-triangle mesh 333x217 x 50 spp 3.45 -> 2.74.  The ray held
// ahead needs the registers of four waves per SIMD with the overflow path (five, spilling 44 B a
// lane: the instances 41.5).  The first bounce keeps one ray per lane: its camera rays are coherent
// (as shares: the mesh 35.8 ms, the instances 39.1).
template <bool OVF>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(OVF ? 4 : 5)))
k_extend_refill(WfParams W, int cur, PassArgs, PathCount count) {
  __shared__ int32_t s_stack[TPT_WF_STACK * TPT_WF_BLOCK];
  QueueMap qm;
  qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
  LaneStackT<OVF> st{s_stack + threadIdx.x, OVF ? W.gstack + (size_t)gtid() * W.gstack_cap : nullptr, TPT_WF_BLOCK,
                     TPT_WF_STACK};
  begin_extension<false>(W, cur, qm.n, count);
  extend_share(W, cur, GlobalTree{W.S}, st, W.refill);
}

__device__ __forceinline__ void add_radiance(float4* L, int32_t id, f3 c) {
  float4 l = L[id];
  L[id] = make_float4(l.x + c.x, l.y + c.y, l.z + c.z, 0.f);
}

// One vertex of a path: its ray, throughput and random stream before shading; scatter() replaces
// them by the next vertex's.
struct PathVertex {
  f3 o, d, beta;
  float last_pdf;
  uint32_t flags;  // bits 0-7 bounce, bit 8 last bounce non-delta
  RngF32 rng{1};
  __device__ __forceinline__ int bounce() const { return (int)(flags & 0xffu); }
};
// The surface a vertex scatters from.
struct VertexSurface {
  f3 p, ng;
  int kind;
  float4 mp;
  float t;
};
// Shadow rays of a vertex and what they add to the path if they are unoccluded.
struct VertexNee {
  bool env, light;
  f3 env_o, env_d, env_c;
  f3 l_d, l_c;  // the shadow kernel rebuilds the light ray's origin p + eps wi and tmax
  float l_dist;
  uint64_t l_state;  // random stream before the light sample (for the self-occlusion decision)
};

// Miss, Russian roulette, emission and next-event estimation at hit h (integrator.rs:71-213);
// false when the path ends here.  gather(c) receives the vertex's own radiance.  ENV_NEE: the
// environment is an image with a non-zero texel, so environment NEE runs.
template <bool ENV_NEE, class Gather>
__device__ __forceinline__ bool shade_vertex(const WfParams& W, const HitRec& h, PathVertex& v, VertexSurface& sf,
                                             VertexNee& nee, Gather gather) {
  if (h.inst == -1) {
    // miss (integrator.rs:71-83); a black map adds nothing, so its paths just end
    if (!W.env.black) {
      f3 bg = W.env.kind == TPT_ENV_IMAGE ? env_lookup32(W.env, v.d) : sky32(v.d);
      f3 c = had(v.beta, bg);
      if (W.env.kind == TPT_ENV_IMAGE && (v.flags & 0x100u)) c = c * mis_weight(v.last_pdf, env_pdf32(W.env, v.d));
      gather(clamp_luminance(c, (float)TPT_FIREFLY_CLAMP));
    }
    return false;
  }
  if (v.bounce() >= W.rr_start) {  // integrator.rs:89-95
    float q = fmaxf(fminf(fmaxf(fmaxf(v.beta.x, v.beta.y), v.beta.z), 0.95f), 0.05f);
    if (v.rng.uni() > q) return false;
    v.beta = v.beta / q;
  }
  int mat;
  sf.t = __int_as_float(h.t);
  hit_geometry32(W.S, h.inst, h.prim, sf.t, v.o, v.d, &sf.p, &sf.ng, &mat);
  sf.kind = W.mats.kind[mat];
  sf.mp = W.mats.p32[mat];
  const f3 mc = f3of(sf.mp), p = sf.p;
  if (sf.kind == TPT_MAT_DIFFUSE_LIGHT) {  // integrator.rs:100-104
    gather(clamp_luminance(had(v.beta, mc), (float)TPT_FIREFLY_CLAMP));
    return false;
  }
  if (mat_is_delta(sf.kind)) return true;
  f3 n_o = dot(sf.ng, v.d) < 0.f ? sf.ng : -sf.ng;  // oriented_normal (integrator.rs:138-140)
  f3 wo = vnorm(-v.d);
  // nee_environment (integrator.rs:148-172); a black map contributes nothing, so the
  // FP32 form skips it (its own random streams need not follow the reference's draws)
  if (ENV_NEE) {
    f3 wi, li;
    float pdf_env;
    env_sample32(W.env, v.rng, &wi, &li, &pdf_env);
    float cs = fmaxf(dot(n_o, wi), 0.f);
    if (cs > 0.f && pdf_env > 0.f && (li.x != 0.f || li.y != 0.f || li.z != 0.f)) {
      f3 f;
      float pdf_b;
      bsdf_eval(sf.kind, mc, sf.mp.w, wo, wi, n_o, &f, &pdf_b);
      f3 c = had(had(v.beta, f), li) * (cs * mis_weight(pdf_env, pdf_b) / pdf_env);
      if (c.x != 0.f || c.y != 0.f || c.z != 0.f) {
        nee.env_o = p + (float)TPT_RAY_EPSILON * wi;
        nee.env_d = wi;
        nee.env_c = c;
        nee.env = true;
      }
    }
  }
  LightSample32 ls;  // nee_area_light (integrator.rs:178-213)
  const uint64_t light_state = v.rng.p.state;
  if (sample_light32(W.lights, v.rng, p, &ls)) {
    f3 to_light = ls.pos - p;
    float dist = sqrtf(dot(to_light, to_light));
    if (dist > 1e-6f) {
      f3 wi = to_light / dist;
      float cs = fmaxf(dot(n_o, wi), 0.f);
      if (cs > 0.f) {
        f3 f;
        float pdf_b;
        bsdf_eval(sf.kind, mc, sf.mp.w, wo, wi, n_o, &f, &pdf_b);
        f3 c = had(had(v.beta, f), ls.emit) * (cs * mis_weight(ls.pdf, pdf_b) / ls.pdf);
        if (c.x != 0.f || c.y != 0.f || c.z != 0.f) {
          nee.l_d = wi;
          nee.l_c = c;
          nee.l_dist = dist;
          nee.l_state = light_state;
          nee.light = true;
        }
      }
    }
  }
  return true;
}

// BSDF sampling: v becomes the next vertex's ray; false when the path ends.
__device__ __forceinline__ bool scatter_vertex(const WfParams& W, const VertexSurface& sf, PathVertex& v) {
  if (v.bounce() + 1 >= W.max_bounces) return false;  // the scattered ray of the last bounce is never traced
  BsdfSample<float> bs;
  if (!bsdf_sample(sf.kind, f3of(sf.mp), sf.mp.w, v.d, sf.p, sf.ng, sf.t, v.rng, &bs)) return false;
  v.beta = had(v.beta, bs.weight);
  v.o = bs.o;
  v.d = bs.d;
  v.last_pdf = bs.pdf;
  v.flags = (uint32_t)(v.bounce() + 1) | (bs.is_delta ? 0u : 0x100u);
  return true;
}

__device__ __forceinline__ void load_vertex(const PathState& ps, int cur, uint32_t slot, PathVertex* v, int32_t* id) {
  const float4 o4 = ps.o[cur][slot], d4 = ps.d[cur][slot], b4 = ps.beta[cur][slot];
  v->o = f3of(o4);
  v->d = f3of(d4);
  v->beta = f3of(b4);
  *id = __float_as_int(b4.w);
  v->last_pdf = o4.w;
  v->flags = __float_as_uint(d4.w);
  v->rng.p.state = ps.rng[cur][slot];
}

// Queue positions of a block's entries in three queues, in LDS: each wave counts its entries, one
// thread a queue (of another wave each) reserves the block's total, and every lane finds its
// position.  k_shade waited for a reservation's way to memory and back, and for three barriers,
// once per queue; now the NEE queues' reservations are under way while the BSDF is sampled, the
// entries are written while the survivors' is, and a turn has three barriers.  Cornell 512^2 x
// 256 spp 21.48 -> 21.21 ms, the 1.31M-triangle mesh 1080p x 32 spp 33.2 -> 32.8, 4096 instances
// adaptive 37.9 -> 37.6 (at five waves per SIMD, with spills, 21.3, 36.3 and 41.9).
static_assert(TPT_WF_BLOCK > 128, "threads 0, 64 and 128 reserve");
struct SlotWords {
  uint32_t n[3][TPT_WF_BLOCK / 64], first[3];
  __device__ __forceinline__ void count(int q, bool pred) {
    const uint64_t mask = __ballot(pred);
    if (__lane_id() == 0) n[q][threadIdx.x >> 6] = (uint32_t)__popcll(mask);
  }
  __device__ __forceinline__ uint32_t reserve(int q, const PathState& ps, int queue) const {
    uint32_t tot = 0;
    for (uint32_t w = 0; w < TPT_WF_BLOCK / 64; w++) tot += n[q][w];
    return tot ? atomicAdd(ps.counters + TPT_CNT_IDX(queue, blockIdx.x & (TPT_WF_SEGS - 1)), tot) : 0u;
  }
  // The slot of a lane with an entry (mask: its wave's lanes with one), or UINT32_MAX as seg_slot.
  __device__ __forceinline__ uint32_t slot(int q, uint64_t mask, const PathState& ps) const {
    uint32_t pos = first[q] + (uint32_t)__popcll(mask & ((1ull << __lane_id()) - 1ull));
    for (uint32_t w = 0; w < threadIdx.x >> 6; w++) pos += n[q][w];
    if (pos >= ps.seg_cap) {
      ps.counters[TPT_CNT_OVERFLOW] = 1u;
      return UINT32_MAX;
    }
    return (blockIdx.x & (TPT_WF_SEGS - 1)) * ps.seg_cap + pos;
  }
};

// ENV_NEE: see shade_vertex (the variant without it needs fewer registers).  GEN: the first
// bounce; path i (position i) is regenerated from its pixel and sample, as k_extend traced it,
// and its radiance sum L[i] is written rather than added to.
template <bool ENV_NEE, bool GEN>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_shade(WfParams W, int cur, PassArgs A) {
  __shared__ SlotWords s_slot[2];  // by turns: a wave may be a turn ahead of the block's slowest
  uint32_t turn = 0;
  QueueMap qm;
  uint32_t n;
  if constexpr (GEN) {
    n = A.n_paths;
  } else {
    qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
    n = qm.n;
  }
  const int nxt = cur ^ 1;
  const uint32_t stride = gridDim.x * blockDim.x;
  for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += stride) {
    const uint32_t i = base + threadIdx.x;
    // path state (valid when i < n)
    PathVertex v;
    v.o = v.d = v.beta = mk(0.f, 0.f, 0.f);
    v.last_pdf = 0.f;
    v.flags = 0;
    int32_t id = 0;
    HitRec h{0, -1, 0};
    if (i < n) {
      if constexpr (GEN) {
        gen_path(W, A, i, &v.rng, &v.o, &v.d);
        v.beta = mk(1.f, 1.f, 1.f);
        id = (int32_t)i;
      } else {
        load_vertex(W.ps, cur, qm.slot(i), &v, &id);
      }
      h = W.ps.hit[i];
    }
    // radiance of this bounce: added to L[id], or (first bounce) gathered and written once
    f3 l0 = mk(0.f, 0.f, 0.f);
    auto gather = [&](f3 c) {
      if constexpr (GEN) l0 = l0 + c;
      else add_radiance(W.ps.L, id, c);
    };
    VertexSurface sf;
    sf.p = sf.ng = mk(0.f, 0.f, 0.f);
    sf.kind = 0;
    sf.mp = make_float4(0.f, 0.f, 0.f, 0.f);
    sf.t = 0.f;
    VertexNee nee;
    nee.env = nee.light = false;
    nee.env_o = nee.env_d = nee.env_c = nee.l_d = nee.l_c = mk(0.f, 0.f, 0.f);
    nee.l_dist = 0.f;
    nee.l_state = 0;
    bool go = false;  // hit a scattering surface: sample the BSDF
    if (i < n) go = shade_vertex<ENV_NEE>(W, h, v, sf, nee, gather);
    if (GEN && i < n) W.ps.L[id] = make_float4(l0.x, l0.y, l0.z, 0.f);
    // the queue positions: the NEE entries' reservations are under way while the BSDF is sampled
    SlotWords& sw = s_slot[turn];
    turn ^= 1;
    if (ENV_NEE) sw.count(0, nee.env);
    sw.count(1, nee.light);
    __syncthreads();
    uint32_t first = 0;  // of the queue that this thread reserves in
    if (ENV_NEE && threadIdx.x == 64) first = sw.reserve(0, W.ps, TPT_CNT_SH);
    if (threadIdx.x == 0) first = sw.reserve(1, W.ps, TPT_CNT_SHL);
    // BSDF sampling; survivors go densely into the next buffer set
    const bool alive = go && scatter_vertex(W, sf, v);
    sw.count(2, alive);
    if (ENV_NEE && threadIdx.x == 64) sw.first[0] = first;
    if (threadIdx.x == 0) sw.first[1] = first;
    __syncthreads();
    if (threadIdx.x == 128) sw.first[2] = sw.reserve(2, W.ps, cur ? TPT_CNT_Q0 : TPT_CNT_Q1);
    if (ENV_NEE && nee.env) {
      const uint32_t je = sw.slot(0, __ballot(true), W.ps);
      if (je != UINT32_MAX) {
        W.ps.sh_o[0][je] = make_float4(nee.env_o.x, nee.env_o.y, nee.env_o.z, 1e30f);
        W.ps.sh_d[0][je] = make_float4(nee.env_d.x, nee.env_d.y, nee.env_d.z, __int_as_float(id));
        W.ps.sh_c[0][je] = make_float4(nee.env_c.x, nee.env_c.y, nee.env_c.z, 1.f);
      }
    }
    if (nee.light) {
      const uint32_t jl = sw.slot(1, __ballot(true), W.ps);
      if (jl != UINT32_MAX) {
        W.ps.sh_d[1][jl] = make_float4(nee.l_d.x, nee.l_d.y, nee.l_d.z, __int_as_float(id));
        W.ps.sh_c[1][jl] = make_float4(nee.l_c.x, nee.l_c.y, nee.l_c.z, nee.l_dist);
        W.ps.sh_l[jl] = make_float4(sf.p.x, sf.p.y, sf.p.z, __int_as_float((int32_t)i));  // also for k_light_selfocc
        W.ps.sh_lv[jl] = nee.l_state;
      }
    }
    __syncthreads();
    if (alive) {
      const uint32_t k = sw.slot(2, __ballot(true), W.ps);
      if (k != UINT32_MAX) {
        W.ps.o[nxt][k] = make_float4(v.o.x, v.o.y, v.o.z, v.last_pdf);
        W.ps.d[nxt][k] = make_float4(v.d.x, v.d.y, v.d.z, __uint_as_float(v.flags));
        W.ps.beta[nxt][k] = make_float4(v.beta.x, v.beta.y, v.beta.z, __int_as_float(id));
        W.ps.rng[nxt][k] = v.rng.p.state;
      }
    }
  }
}

// The reference's light shadow ray can be blocked by the light itself; that decision is taken
// in FP64 (tpt_selfocc64.h) here, in a kernel of its own so the FP64 registers do not weigh on
// k_shade.  Its inputs are rebuilt with the reference's precision: the shading point by the
// FP64 World::hit of the path's FP32 ray on the primitive it hit (the ray from the path queue,
// or, on the first bounce, the camera ray generated again), the light and its 53-bit uniforms
// drawn again from the stream state saved before the light sample.  The slots of the rays that
// remain go densely into the SHK queue, so k_shadow's waves carry no lanes for dropped rays
// (about 30% on a rectangle light).
template <bool GEN>
__global__ void __launch_bounds__(TPT_WF_BLOCK) k_light_selfocc(WfParams W, int cur, PassArgs A,
                                                                 PathCount count) {
  __shared__ uint32_t s_slot[8];
  tell_count(W, count);
  QueueMap qm, qp;
  qm.load(W.ps.counters, TPT_CNT_SHL, W.ps.seg_cap);
  if constexpr (!GEN) qp.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
  const uint32_t n = qm.n;
  uint32_t dropped = 0;  // self-occluded samples this thread saw
  for (uint32_t base = blockIdx.x * blockDim.x; base < n; base += gridDim.x * blockDim.x) {
    const uint32_t j = base + threadIdx.x;
    uint32_t slot = 0;
    bool keep = false;
    if (j < n) {
      slot = qm.slot(j);
      const float4 l = W.ps.sh_l[slot];
      // the light and its uniforms first: their loads overlap the hit point's chain below
      RngF32 rng(1);
      rng.p.state = W.ps.sh_lv[slot];
      const int idx = light_pick32(W.lights, rng);
      const double u = rng.uni53(), v = rng.uni53();
      const uint32_t pos = (uint32_t)__float_as_int(l.w);  // the path's dense position this bounce
      f3 o, d;
      if constexpr (GEN) {
        RngF32 cam(1);
        gen_path(W, A, pos, &cam, &o, &d);
      } else {
        const uint32_t ps = qp.slot(pos);
        o = f3of(W.ps.o[cur][ps]);
        d = f3of(W.ps.d[cur][ps]);
      }
      const HitRec hr = W.ps.hit[pos];
      const D3 p64 = hit_point64(W.S64, W.S.tri_orig, hr.inst, hr.prim, o, d, f3of(l));
      keep = !light_self_occluded64(W.S64, W.lights, idx, p64, u, v);
    }
    const uint32_t k = seg_slot(keep, W.ps, TPT_CNT_SHK, s_slot);  // every thread of the block
    if (keep && k != UINT32_MAX) W.ps.shl_keep[k] = slot;
    if (j < n && !keep) dropped++;
  }
  for (int off = 32; off > 0; off >>= 1) dropped += (uint32_t)__shfl_down((int)dropped, off);
  uint64_t* st = W.ps.stats + (blockIdx.x & (TPT_WF_SEGS - 1)) * TPT_STAT_STRIDE;
  if (__lane_id() == 0 && dropped) atomicAdd((unsigned long long*)&st[4], (unsigned long long)dropped);
  if (gtid() == 0 && n) atomicAdd((unsigned long long*)&W.ps.stats[3], (unsigned long long)n);
}

// Any hit for one shadow queue (0: environment, 1: area light); an unoccluded ray adds its
// contribution to its path's radiance.  A path has at most one ray per queue, so the
// read-modify-write of L[id] has a single writer per launch.
template <bool OVF>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(5))) k_shadow(WfParams W, int queue, PathCount count) {
  tell_count(W, count);
  __shared__ int32_t s_stack[TPT_WF_STACK * TPT_WF_BLOCK];
  QueueMap qm;
  qm.load(W.ps.counters, queue ? TPT_CNT_SHK : TPT_CNT_SH, W.ps.seg_cap);
  const float4* __restrict__ qo = queue ? W.ps.sh_l : W.ps.sh_o[0];
  const float4* __restrict__ qd = W.ps.sh_d[queue];
  const float4* __restrict__ qc = W.ps.sh_c[queue];
  LaneStackT<OVF> st{s_stack + threadIdx.x, OVF ? W.gstack + (size_t)gtid() * W.gstack_cap : nullptr, TPT_WF_BLOCK,
                     TPT_WF_STACK};
  uint32_t traced = 0;
  for (uint32_t j = gtid(); j < qm.n; j += gridDim.x * blockDim.x) {
    const uint32_t slot = queue ? W.ps.shl_keep[qm.slot(j)] : qm.slot(j);
    const float4 o4 = qo[slot], d4 = qd[slot];
    f3 o = f3of(o4);
    float tmax = o4.w;
    if (queue) {  // light queue: o4 is the shading point, sh_c's w the distance to the light sample
      o = o + (float)TPT_RAY_EPSILON * f3of(d4);
      tmax = light_shadow_tmax32(qc[slot].w);
    }
    HitF32 h;
    traced++;
    // the contribution is read only for an unoccluded ray, after the traversal
    if (!trace_f32<true>(W.S, o, f3of(d4), (float)TPT_RAY_EPSILON, tmax, &h, st))
      add_radiance(W.ps.L, __float_as_int(d4.w), f3of(qc[slot]));
  }
  // one atomic per wave for the shadow-ray count
  uint32_t tot = traced;
  for (int off = 32; off > 0; off >>= 1) tot += (uint32_t)__shfl_down((int)tot, off);
  if (__lane_id() == 0 && tot)
    atomicAdd((unsigned long long*)&W.ps.stats[(blockIdx.x & (TPT_WF_SEGS - 1)) * TPT_STAT_STRIDE + 1],
              (unsigned long long)tot);
}

// The shadow rays of a wave's share, as extend_share: a lane's next ray is loaded one start ahead
// (the light queue's list of surviving slots two ahead), and the radiance of the rays that were
// found unoccluded is added when the next rays start, so that the wave waits for that read once for
// many rays.
template <class Tree, class Stack>
__device__ __forceinline__ void shadow_share(const WfParams& W, int queue, const Tree& tree, const Stack& st, int lanes) {
  QueueMap qm;
  qm.load(W.ps.counters, queue ? TPT_CNT_SHK : TPT_CNT_SH, W.ps.seg_cap);
  const uint32_t n = qm.n;
  const float4* __restrict__ qo = queue ? W.ps.sh_l : W.ps.sh_o[0];
  const float4* __restrict__ qd = W.ps.sh_d[queue];
  const float4* __restrict__ qc = W.ps.sh_c[queue];
  WaveShare share;
  TraceF32<true, Tree> tr;
  uint32_t traced = 0;
  bool live = false, lit = false;  // lit: the lane's last ray was unoccluded, its radiance is still to be added
  uint32_t slot = 0;
  int32_t id = 0;
  // the next ray: its slot, origin, direction, tmax (light queue: distance to the light sample)
  uint32_t nslot = 0, far_slot;
  bool have, have_far;
  float4 no = make_float4(0.f, 0.f, 0.f, 0.f), nd = no;
  float ndist = 0.f;
  auto fetch_slot = [&](bool want) {  // the slot of the ray after the next
    const uint32_t t = share.take(want);
    if (want) {
      have_far = t < n;
      if (have_far) far_slot = queue ? W.ps.shl_keep[qm.slot(t)] : qm.slot(t);
    }
  };
  auto fetch_ray = [&](bool want) {
    if (!want) return;
    have = have_far;
    nslot = far_slot;
    if (have) {
      no = qo[nslot];
      nd = qd[nslot];
      ndist = queue ? qc[nslot].w : no.w;
    }
  };
  have_far = have = false;
  far_slot = 0;
  fetch_slot(true);
  fetch_ray(true);
  fetch_slot(true);
  for (;;) {
    const int nl = __popcll(__ballot(live));
    const bool some = __ballot(!live && have) != 0;
    if (nl == 0 || (some && nl < lanes)) {  // wave-uniform
      const bool start = !live && have;
      const bool add = !live && lit;
      float4 l, c;
      if (add) {
        l = W.ps.L[id];
        c = qc[slot];
      }
      const int32_t add_id = id;
      if (start) {
        slot = nslot;
        id = __float_as_int(nd.w);
        f3 o = f3of(no);
        float tmax = ndist;
        if (queue) {  // the queue holds the shading point and the distance to the light sample
          o = o + (float)TPT_RAY_EPSILON * f3of(nd);
          tmax = light_shadow_tmax32(ndist);
        }
        traced++;
        live = tr.init(W.S, o, f3of(nd), (float)TPT_RAY_EPSILON, tmax);
        have = false;
      }
      if (add) {
        W.ps.L[add_id] = make_float4(l.x + c.x, l.y + c.y, l.z + c.z, 0.f);
        lit = false;
      }
      if (start && !live) lit = !tr.found;
      const bool want = !have;
      fetch_ray(want);
      fetch_slot(want);
      if (!some) break;  // nothing was started: the share is taken
      continue;
    }
    if (live && !tr.step(W.S, st, tree)) {
      lit = !tr.found;
      live = false;
    }
  }
  uint32_t tot = traced;
  for (int off = 32; off > 0; off >>= 1) tot += (uint32_t)__shfl_down((int)tot, off);
  if (__lane_id() == 0 && tot)
    atomicAdd((unsigned long long*)&W.ps.stats[(blockIdx.x & (TPT_WF_SEGS - 1)) * TPT_STAT_STRIDE + 1],
              (unsigned long long)tot);
}

// k_shadow for small scenes, see k_extend_small.
// Cornell 512^2 x 256 spp 22.3 -> 21.5 ms; the look-ahead needs the registers of four
// waves per SIMD (at five, with spills, 22.0; at six 23.0); rays started below 57 tracing lanes 22.5,
// 33 and 9 within 0.3% of 17 (TPT_SMALL_LANES_SH).
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_shadow_small(WfParams W, int queue, PathCount count) {
  extern __shared__ float4 s_small[];
  tell_count(W, count);
  LaneStackT<false> st;
  const SmallTree tree = load_small<TPT_WF_BLOCK>(W.S, W.small, s_small, &st);
  shadow_share(W, queue, tree, st, TPT_SMALL_LANES_SH);
}

// k_shadow for deep trees, see k_extend_refill.
template <bool OVF>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(4)))
k_shadow_refill(WfParams W, int queue, PathCount count) {
  tell_count(W, count);
  __shared__ int32_t s_stack[TPT_WF_STACK * TPT_WF_BLOCK];
  LaneStackT<OVF> st{s_stack + threadIdx.x, OVF ? W.gstack + (size_t)gtid() * W.gstack_cap : nullptr, TPT_WF_BLOCK,
                     TPT_WF_STACK};
  shadow_share(W, queue, GlobalTree{W.S}, st, W.refill);
}

// The trees k_tail walks and this lane's stack, in `mem`.
template <class Tree, bool OVF>
__device__ __forceinline__ Tree tail_tree(const WfParams& W, float4* mem, LaneStackT<OVF>* st) {
  if constexpr (Tree::kWorldOnly) {
    return load_small<TPT_WF_BLOCK>(W.S, W.small, mem, st);
  } else {
    *st = LaneStackT<OVF>{reinterpret_cast<int32_t*>(mem) + threadIdx.x,
                          OVF ? W.gstack + (size_t)gtid() * W.gstack_cap : nullptr, TPT_WF_BLOCK, TPT_WF_STACK};
    return GlobalTree{W.S};
  }
}

// The rest of a few paths in one launch: each lane walks its path to the end -- extension, shading,
// the light self-occlusion decision, shadow rays and scattering by the same functions as the
// kernels above, contributions added in their order, so a path's radiance is the same bit for bit.
// Tree: SmallTree for small scenes (64^2 x 4 spp of the Cornell box 245 -> 233 us per render, the same
// rays on device memory).  GEN: the whole paths of a small pass (camera rays generated here);
// otherwise the paths of queue cur, whose hits this bounce's extension has stored.
template <class Tree, bool OVF, bool ENV_NEE, bool GEN>
__global__ void __launch_bounds__(TPT_WF_BLOCK) __attribute__((amdgpu_waves_per_eu(2)))
k_tail(WfParams W, int cur, PassArgs A) {
  extern __shared__ float4 s_small[];
  LaneStackT<OVF> st;
  const Tree tree = tail_tree<Tree>(W, s_small, &st);
  QueueMap qm;
  uint32_t n;
  if constexpr (GEN) {
    n = A.n_paths;
  } else {
    qm.load(W.ps.counters, cur ? TPT_CNT_Q1 : TPT_CNT_Q0, W.ps.seg_cap);
    n = qm.n;
  }
  const uint32_t lanes = lanes_per_wave(n);
  uint32_t next = (gtid() >> 6) * lanes + __lane_id();
  if (__lane_id() >= lanes) next = n;
  uint32_t n_ext = 0, n_sh = 0, n_light = 0, n_drop = 0;
  bool alive = false;
  PathVertex v;
  int32_t id = 0;
  f3 L = mk(0.f, 0.f, 0.f);
  for (;;) {
    HitRec h;
    bool have_hit = false;
    if (!alive) {
      if (next >= n) break;
      if constexpr (GEN) {
        gen_path(W, A, next, &v.rng, &v.o, &v.d);
        v.beta = mk(1.f, 1.f, 1.f);
        v.last_pdf = 0.f;
        v.flags = 0;
        id = (int32_t)next;
        L = mk(0.f, 0.f, 0.f);
      } else {
        load_vertex(W.ps, cur, qm.slot(next), &v, &id);
        h = W.ps.hit[next];
        have_hit = true;
        L = f3of(W.ps.L[id]);
      }
      next += gridDim.x * (TPT_WF_BLOCK / 64) * lanes;
      alive = true;
    }
    if (!have_hit) {
      HitF32 t;
      trace_f32<false>(W.S, tree, v.o, v.d, (float)TPT_RAY_EPSILON, 1e30f, &t, st);
      h = HitRec{__float_as_int(t.t), t.inst, t.prim};
      n_ext++;
    }
    VertexSurface sf;
    VertexNee nee;
    nee.env = nee.light = false;
    alive = shade_vertex<ENV_NEE>(W, h, v, sf, nee, [&](f3 c) { L = L + c; });
    if (nee.light) {  // k_light_selfocc, then k_shadow on the light queue
      n_light++;
      RngF32 rng(1);
      rng.p.state = nee.l_state;
      const int idx = light_pick32(W.lights, rng);
      const double lu = rng.uni53(), lv = rng.uni53();
      const D3 p64 = hit_point64(W.S64, W.S.tri_orig, h.inst, h.prim, v.o, v.d, sf.p);
      if (light_self_occluded64(W.S64, W.lights, idx, p64, lu, lv)) {
        n_drop++;
      } else {
        HitF32 t;
        n_sh++;
        if (!trace_f32<true>(W.S, tree, sf.p + (float)TPT_RAY_EPSILON * nee.l_d, nee.l_d, (float)TPT_RAY_EPSILON,
                             light_shadow_tmax32(nee.l_dist), &t, st))
          L = L + nee.l_c;
      }
    }
    if (ENV_NEE && nee.env) {  // k_shadow on the environment queue
      HitF32 t;
      n_sh++;
      if (!trace_f32<true>(W.S, tree, nee.env_o, nee.env_d, (float)TPT_RAY_EPSILON, 1e30f, &t, st)) L = L + nee.env_c;
    }
    alive = alive && scatter_vertex(W, sf, v);
    if (!alive) W.ps.L[id] = make_float4(L.x, L.y, L.z, 0.f);
  }
  for (int off = 32; off > 0; off >>= 1) {
    n_ext += (uint32_t)__shfl_down((int)n_ext, off);
    n_sh += (uint32_t)__shfl_down((int)n_sh, off);
    n_light += (uint32_t)__shfl_down((int)n_light, off);
    n_drop += (uint32_t)__shfl_down((int)n_drop, off);
  }
  if (__lane_id() == 0 && (n_ext | n_sh | n_light)) {
    unsigned long long* stat = (unsigned long long*)W.ps.stats + (blockIdx.x & (TPT_WF_SEGS - 1)) * TPT_STAT_STRIDE;
    atomicAdd(&stat[0], (unsigned long long)n_ext);
    atomicAdd(&stat[1], (unsigned long long)n_sh);
    atomicAdd(&stat[3], (unsigned long long)n_light);
    atomicAdd(&stat[4], (unsigned long long)n_drop);
    atomicAdd(&stat[5], (unsigned long long)n_ext);
  }
}

// Non-adaptive: pixel p accumulates the k paths of this pass, in sample order.
__global__ void __launch_bounds__(TPT_WF_BLOCK) k_accumulate(WfParams W, AccumArgs A) {
  for (uint32_t p = gtid(); p < A.n_pixels; p += gridDim.x * blockDim.x) {
    double r = 0, g = 0, b = 0, r2 = 0, g2 = 0, b2 = 0;
    uint32_t first, step;
    path_index(p, A.n_pixels, A.k, &first, &step);
    for (uint32_t j = 0; j < A.k; j++) {
      float4 l = W.ps.L[first + j * step];
      double x = l.x, y = l.y, z = l.z;
      r += x; g += y; b += z;
      r2 += x * x; g2 += y * y; b2 += z * z;
    }
    uint32_t g_pix = A.pixel0 + p;
    A.acc[3 * g_pix] += r; A.acc[3 * g_pix + 1] += g; A.acc[3 * g_pix + 2] += b;
    A.acc_w[g_pix] += (double)A.k;
    if (A.acc_sq) { A.acc_sq[3 * g_pix] += r2; A.acc_sq[3 * g_pix + 1] += g2; A.acc_sq[3 * g_pix + 2] += b2; }
  }
  if (gtid() == 0) atomicAdd((unsigned long long*)&W.ps.stats[2], (unsigned long long)A.n_pixels * A.k);
}

// Adaptive (render.rs:143-179): for each active pixel take its k new samples in sample order,
// Welford on luminance, stop at the reference's criterion; samples past the stop are dropped.
// Survivors are compacted into `active_out`.
__global__ void __launch_bounds__(TPT_WF_BLOCK) k_accumulate_adaptive(WfParams W, AdaptiveArgs A) {
  __shared__ uint32_t s_slot[8];
  const uint32_t stride = gridDim.x * blockDim.x;
  uint32_t kept = 0;  // samples this thread added to its pixels (the paths the render counts)
  for (uint32_t base = blockIdx.x * blockDim.x; base < A.n_active; base += stride) {
    uint32_t j = base + threadIdx.x;
    bool keep = false;
    int32_t pix = 0;
    if (j < A.n_active) {
      pix = A.active_in[j];
      uint32_t n = A.nsamp[pix];
      const uint32_t n0 = n;
      double mean = A.welford[2 * pix], m2 = A.welford[2 * pix + 1];
      double r = 0, g = 0, b = 0, r2 = 0, g2 = 0, b2 = 0;
      bool stop = false;
      uint32_t first, step;
      path_index(j, A.n_active, A.k, &first, &step);
      for (uint32_t k = 0; k < A.k && !stop; k++) {
        float4 l = W.ps.L[first + k * step];
        double x = l.x, y = l.y, z = l.z;
        r += x; g += y; b += z;
        r2 += x * x; g2 += y * y; b2 += z * z;
        n += 1;
        double lum = 0.2126 * x + 0.7152 * y + 0.0722 * z;
        double delta = lum - mean;
        mean += delta / (double)n;
        double delta2 = lum - mean;
        m2 += delta * delta2;
        if (n >= A.min_spp) {
          double var = n > 1 ? m2 / (double)(n - 1) : __longlong_as_double(0x7ff0000000000000ll);
          double rel = sqrt(var) / fmax(fabs(mean), 1e-4);
          if (rel < A.threshold) stop = true;
        }
        if (n >= A.max_spp) stop = true;
      }
      A.acc[3 * pix] += r; A.acc[3 * pix + 1] += g; A.acc[3 * pix + 2] += b;
      if (A.acc_sq) { A.acc_sq[3 * pix] += r2; A.acc_sq[3 * pix + 1] += g2; A.acc_sq[3 * pix + 2] += b2; }
      A.acc_w[pix] = (double)n;
      A.nsamp[pix] = n;
      kept += n - n0;
      A.welford[2 * pix] = mean;
      A.welford[2 * pix + 1] = m2;
      keep = !stop;
    }
    const uint32_t q = block_slot(keep, A.n_active_out, s_slot);
    if (keep) A.active_out[q] = pix;
  }
  for (int off = 32; off > 0; off >>= 1) kept += (uint32_t)__shfl_down((int)kept, off);
  if (__lane_id() == 0 && kept)
    atomicAdd((unsigned long long*)&W.ps.stats[(blockIdx.x & (TPT_WF_SEGS - 1)) * TPT_STAT_STRIDE + 2],
              (unsigned long long)kept);
}

// ---------------------------------------------------------------- host-side launchers
// Grid of at most TPT_WF_MAX_BLOCKS blocks: the kernels loop over their queues, so the grid only
// needs to fill the chip (256 CUs x 8 blocks); larger grids cost dispatch time per bounce,
// most of all for launches whose queues have shrunk to a few paths.
// The grid is a multiple of TPT_WF_SEGS (queue segments follow blockIdx % TPT_WF_SEGS).
static inline uint32_t grid_for(uint32_t n) {
  uint32_t b = (n + TPT_WF_BLOCK - 1) / TPT_WF_BLOCK;
  b = (b + TPT_WF_SEGS - 1) / TPT_WF_SEGS * TPT_WF_SEGS;
  return b < TPT_WF_SEGS ? TPT_WF_SEGS : (b > TPT_WF_MAX_BLOCKS ? TPT_WF_MAX_BLOCKS : b);
}

// Blocks of `kernel` that are resident on the whole device at once (CUs x blocks per CU at the
// kernel's register and LDS use), rounded down to a multiple of TPT_WF_SEGS.  A grid-stride
// kernel launched with more blocks than this runs its last blocks after the first ones finish,
// with the device partly idle (5 resident blocks per CU against 8 launched leaves a 60 %-full
// second round); capping the grid at the resident count gives every block the same share.
static uint32_t resident_blocks(const void* kernel, uint32_t lds = 0) {
  static std::mutex mu;
  static std::map<std::pair<const void*, uint32_t>, uint32_t> cache;  // one device model per process
  std::lock_guard<std::mutex> lock(mu);
  auto it = cache.find({kernel, lds});
  if (it != cache.end()) return it->second;
  int dev = 0, cus = 0, per_cu = 0;
  uint32_t r = TPT_WF_MAX_BLOCKS;
  if (hipGetDevice(&dev) == hipSuccess &&
      hipDeviceGetAttribute(&cus, hipDeviceAttributeMultiprocessorCount, dev) == hipSuccess &&
      hipOccupancyMaxActiveBlocksPerMultiprocessor(&per_cu, kernel, TPT_WF_BLOCK, lds) == hipSuccess && cus > 0 &&
      per_cu > 0) {
    r = (uint32_t)cus * (uint32_t)per_cu / TPT_WF_SEGS * TPT_WF_SEGS;
    r = std::max<uint32_t>(TPT_WF_SEGS, std::min<uint32_t>(r, TPT_WF_MAX_BLOCKS));
  }
  cache[{kernel, lds}] = r;
  return r;
}

// lds: bytes of LDS that the launch adds to the kernel's own.
static inline dim3 grid_of(uint32_t n, const void* kernel, uint32_t lds = 0) {
  return dim3(std::min(grid_for(n), resident_blocks(kernel, lds)));
}
static inline uint32_t small_lds(const WfParams& W) { return small_lds(W.small, TPT_WF_BLOCK); }

hipError_t wf_launch_clear_radiance(const WfParams& W, uint32_t n, hipStream_t s) {
  hipLaunchKernelGGL(k_clear_radiance, dim3(grid_for(n)), dim3(TPT_WF_BLOCK), 0, s, W, n);
  return hipGetLastError();
}
// Extension launches, timed by events that the dispatch records itself when ev0 is given.
template <class K>
static void launch_timed(K kernel, uint32_t max_n, hipStream_t s, hipEvent_t ev0, hipEvent_t ev1, const WfParams& W,
                         int cur, const PassArgs& A, const PathCount& count, uint32_t lds = 0) {
  const dim3 grid = grid_of(max_n, (const void*)kernel, lds);
  if (ev0) hipExtLaunchKernelGGL(kernel, grid, dim3(TPT_WF_BLOCK), lds, s, ev0, ev1, 0, W, cur, A, count);
  else hipLaunchKernelGGL(kernel, grid, dim3(TPT_WF_BLOCK), lds, s, W, cur, A, count);
}
hipError_t wf_launch_extend(const WfParams& W, int cur, const PassArgs* gen, const PathCount& count, uint32_t max_n,
                            hipStream_t s, hipEvent_t ev0, hipEvent_t ev1) {
  const PassArgs A = gen ? *gen : PassArgs{};
  auto launch = [&](auto kernel) { launch_timed(kernel, max_n, s, ev0, ev1, W, cur, A, count); };
  if (W.small.bytes > 0) {
    const uint32_t lds = small_lds(W);
    if (gen) launch_timed(k_extend_small<true>, max_n, s, ev0, ev1, W, cur, A, count, lds);
    else launch_timed(k_extend_small<false>, max_n, s, ev0, ev1, W, cur, A, count, lds);
  } else if (!gen && W.refill > 0) {
    W.gstack ? launch(k_extend_refill<true>) : launch(k_extend_refill<false>);
  } else {
    if (W.gstack) gen ? launch(k_extend<true, true>) : launch(k_extend<true, false>);
    else gen ? launch(k_extend<false, true>) : launch(k_extend<false, false>);
  }
  return hipGetLastError();
}
template <class Tree, bool OVF, bool ENV_NEE>
static void launch_tail(const WfParams& W, int cur, const PassArgs* gen, uint32_t n, hipStream_t s) {
  const PassArgs A = gen ? *gen : PassArgs{};
  const uint32_t lds = Tree::kWorldOnly ? small_lds(W) : TPT_WF_STACK * TPT_WF_BLOCK * 4;
  auto launch = [&](auto kernel) {
    const uint32_t waves = (n + TPT_WF_MIN_LANES - 1) / TPT_WF_MIN_LANES;
    hipLaunchKernelGGL(kernel, grid_of(std::min(waves, 1u << 20) * 64, (const void*)kernel, lds), dim3(TPT_WF_BLOCK), lds,
                       s, W, cur, A);
  };
  if (gen) launch(k_tail<Tree, OVF, ENV_NEE, true>);
  else launch(k_tail<Tree, OVF, ENV_NEE, false>);
}
static inline bool env_nee(const WfParams& W) { return W.env.kind == TPT_ENV_IMAGE && !W.env.black; }
hipError_t wf_launch_tail(const WfParams& W, int cur, const PassArgs* gen, uint32_t n, hipStream_t s) {
  const bool env = env_nee(W);
  if (W.small.bytes > 0)
    env ? launch_tail<SmallTree, false, true>(W, cur, gen, n, s) : launch_tail<SmallTree, false, false>(W, cur, gen, n, s);
  else if (W.gstack)
    env ? launch_tail<GlobalTree, true, true>(W, cur, gen, n, s) : launch_tail<GlobalTree, true, false>(W, cur, gen, n, s);
  else
    env ? launch_tail<GlobalTree, false, true>(W, cur, gen, n, s) : launch_tail<GlobalTree, false, false>(W, cur, gen, n, s);
  return hipGetLastError();
}
template <bool ENV_NEE, bool GEN>
static void launch_shade(const WfParams& W, int cur, const PassArgs& A, uint32_t max_n, hipStream_t s) {
  hipLaunchKernelGGL((k_shade<ENV_NEE, GEN>), grid_of(max_n, (const void*)k_shade<ENV_NEE, GEN>), dim3(TPT_WF_BLOCK), 0,
                     s, W, cur, A);
}
hipError_t wf_launch_shade(const WfParams& W, int cur, const PassArgs* gen, uint32_t max_n, hipStream_t s) {
  const PassArgs A = gen ? *gen : PassArgs{};
  if (env_nee(W)) {
    if (gen) launch_shade<true, true>(W, cur, A, max_n, s);
    else launch_shade<true, false>(W, cur, A, max_n, s);
  } else {
    if (gen) launch_shade<false, true>(W, cur, A, max_n, s);
    else launch_shade<false, false>(W, cur, A, max_n, s);
  }
  return hipGetLastError();
}
hipError_t wf_launch_light_selfocc(const WfParams& W, int cur, const PassArgs* gen, const PathCount& count,
                                   uint32_t max_n, hipStream_t s) {
  const PassArgs A = gen ? *gen : PassArgs{};
  auto launch = [&](auto kernel) {
    hipLaunchKernelGGL(kernel, grid_of(max_n, (const void*)kernel), dim3(TPT_WF_BLOCK), 0, s, W, cur, A, count);
  };
  gen ? launch(k_light_selfocc<true>) : launch(k_light_selfocc<false>);
  return hipGetLastError();
}
hipError_t wf_launch_shadow(const WfParams& W, int queue, const PathCount& count, uint32_t max_n, hipStream_t s) {
  auto launch = [&](auto kernel, uint32_t lds = 0) {
    hipLaunchKernelGGL(kernel, grid_of(max_n, (const void*)kernel, lds), dim3(TPT_WF_BLOCK), lds, s, W, queue, count);
  };
  if (W.small.bytes > 0) {
    launch(k_shadow_small, small_lds(W));
    return hipGetLastError();
  }
  if (W.refill > 0) W.gstack ? launch(k_shadow_refill<true>) : launch(k_shadow_refill<false>);
  else W.gstack ? launch(k_shadow<true>) : launch(k_shadow<false>);
  return hipGetLastError();
}
hipError_t wf_launch_accumulate(const WfParams& W, const AccumArgs& A, hipStream_t s) {
  hipLaunchKernelGGL(k_accumulate, dim3(grid_for(A.n_pixels)), dim3(TPT_WF_BLOCK), 0, s, W, A);
  return hipGetLastError();
}
hipError_t wf_launch_accumulate_adaptive(const WfParams& W, const AdaptiveArgs& A, hipStream_t s) {
  hipLaunchKernelGGL(k_accumulate_adaptive, dim3(grid_for(A.n_active)), dim3(TPT_WF_BLOCK), 0, s, W, A);
  return hipGetLastError();
}
// Upper bound of the threads of any launch above over n entries (sizes per-thread areas).
uint32_t wf_grid_threads(uint32_t n) {
  return grid_for(std::min(n, 1u << 20) * (64 / TPT_WF_MIN_LANES)) * TPT_WF_BLOCK;
}

}  // namespace tpt
