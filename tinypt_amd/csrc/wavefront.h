// wavefront.h -- parameters of the FP32 wavefront kernels (k_wavefront.hip) and their launchers.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "tpt_kernels.h"
#include "tpt_small32.h"
#include "tpt_trace32.h"

namespace tpt {

#define TPT_WF_BLOCK 256
#define TPT_WF_MAX_BLOCKS 2048
static_assert(TPT_WF_BLOCK % 64 == 0 && TPT_WF_BLOCK / 64 <= 7, "block_slot keeps per-wave counts in 7 LDS words");
#define TPT_WF_STACK 24      // LDS stack entries per lane (24 KB per 256-lane block)
#define TPT_WF_STACK_ADJ 16  // the adjoint kernel keeps 16 in LDS (plus 4 KB of gradient slots)

// Queues are split into TPT_WF_SEGS segments.  A block reserves its entries in segment
// blockIdx % TPT_WF_SEGS -- with grids a multiple of TPT_WF_SEGS, the blocks of one XCD -- with
// one atomic on that segment's counter.  Reservations that all hit one counter (or one cache
// line) serialise at the memory side across the 8 XCDs and throttled the shading kernel; each
// counter therefore sits on a 256 B line of its own.  Consumers see a queue as dense positions
// 0..n-1 running through segment 0, then 1, ... (QueueMap).
#define TPT_WF_SEGS 8
#define TPT_CNT_STRIDE 64  // uint32 words between counters (256 B)
#define TPT_CNT_Q0 0
#define TPT_CNT_Q1 1
#define TPT_CNT_SH 2   // environment shadow queue
#define TPT_CNT_SHL 3  // area-light shadow queue
#define TPT_CNT_SHK 4  // slots of the area-light queue entries that the light does not shadow itself
#define TPT_CNT_IDX(q, g) (((q) * TPT_WF_SEGS + (g)) * TPT_CNT_STRIDE)
#define TPT_CNT_ACTIVE (5 * TPT_WF_SEGS * TPT_CNT_STRIDE)    // adaptive active-pixel list (one dense queue)
#define TPT_CNT_OVERFLOW (TPT_CNT_ACTIVE + TPT_CNT_STRIDE)  // set if a segment would overflow (never by construction)
#define TPT_NUM_CNT (TPT_CNT_OVERFLOW + TPT_CNT_STRIDE)
#define TPT_STAT_STRIDE 32  // uint64 words of statistics per segment (256 B)
#define TPT_STAT_WORDS (TPT_WF_SEGS * TPT_STAT_STRIDE)
// Few paths: a bounce's four or five launches take 40 to 300 us however few paths they have (cold
// instruction and scalar caches, the longest traversal of 64 divergent lanes), so k_tail walks the
// last paths to their ends in one launch.  It takes a pass of at most TPT_WF_TAIL_FIRST paths whole
// and the others once at most TPT_WF_TAIL_MAX paths are left.  Measured on MI355X, us per render,
// bounce by bounce / with k_tail: Cornell box of 16K paths 654 / 241, 256K 756 / 445, 512K 842 / 645;
// 20k-triangle mesh of 16K paths 1343 / 452, 256K 2017 / 1181; a whole pass of 1M paths is slower
// (Cornell 1038 / 1098).  Left-over paths: the 1.31M-triangle
// mesh at 1080p x 32 spp 43.0 / 39.5 ms, a 20k-triangle mesh of 3.6M paths 4.09 / 3.49 ms, each within
// 1% for limits of 2^16 to 2^18.
#define TPT_WF_TAIL_FIRST (1u << 18)
#define TPT_WF_TAIL_MAX (1u << 17)
// A bounce is queued before its path count is known if the bounce before it had this many paths:
// a report takes the host about 40 us to act on, which long kernels hide and short ones do not
// (default scene 256^2 x 64 spp: 640 us; waiting for every report 787 us).
#define TPT_WF_AHEAD_MIN (1u << 19)
#define TPT_WF_MIN_LANES 8  // rays a wave takes at least when few rays are spread over the waves
static_assert(TPT_WF_MAX_BLOCKS % TPT_WF_SEGS == 0, "grids are multiples of TPT_WF_SEGS");

// Entries per queue segment for queues of at most P entries.  The shading kernel's block b
// handles input chunks c (TPT_WF_BLOCK positions each) with c = b (mod grid), so with a grid that
// is a multiple of TPT_WF_SEGS a segment receives the outputs of at most ceil(chunks / SEGS)
// chunks.
inline uint32_t wf_seg_cap(uint32_t P) {
  const uint32_t chunks = (P + TPT_WF_BLOCK - 1) / TPT_WF_BLOCK;
  return (chunks + TPT_WF_SEGS - 1) / TPT_WF_SEGS * TPT_WF_BLOCK;
}

// Closest hit of one extension ray: t (float bits), instance code, triangle slot (12 B).
struct HitRec {
  int32_t t, inst, prim;
};

// Path state, structure of arrays, in two buffer sets: the live paths of a bounce sit in the
// segmented queue of one set; shading writes the survivors into the other set, so every kernel
// reads its inputs coalesced.  A path carries its id (the slot of its (pixel, sample) in the
// pass) and gathers radiance in L[id].  hit is indexed by dense queue position.
struct PathState {
  float4* o[2];     // origin xyz, pdf of the last BSDF sample
  float4* d[2];     // direction xyz, flags (bits 0-7 bounce, bit 8 last bounce non-delta)
  float4* beta[2];  // throughput xyz, path id (int bits)
  uint64_t* rng[2];
  HitRec* hit;      // closest hit of queue position i
  float4* L;        // radiance gathered so far, by path id
  // shadow rays, one segmented queue per kind: [0] environment, [1] area light
  float4* sh_o[2];  // environment queue: origin, tmax ([1] unused)
  float4* sh_d[2];  // direction, path id (int bits)
  float4* sh_c[2];  // contribution if unoccluded; w: 1 (environment) or the distance to the light
                    // sample (light; origin p + eps wi and tmax follow from it)
  float4* sh_l;     // light queue: shading point xyz, dense position of the path in its queue (int bits)
  uint64_t* sh_lv;  // light queue: random stream state before the light sample (its light and
                    // 53-bit uniforms are drawn again from it for the self-occlusion test)
  uint32_t* shl_keep;  // segmented queue of light-queue slots whose ray is traced (not self-occluded)
  uint32_t* counters;
  uint64_t* stats;  // per segment g: [g * TPT_STAT_STRIDE + k], k = 0 extension rays, 1 shadow rays, 2 paths,
                    // 3 area-light samples, 4 of them shadowed by their own light, 5 extension rays that
                    // k_tail traced
  uint32_t seg_cap; // entries per queue segment (wf_seg_cap of the allocated path count)
  uint32_t pad;
};

// Dense queue position -> slot of a segmented queue.
struct QueueMap {
  uint32_t pre[TPT_WF_SEGS];  // entries before segment g
  uint32_t n;                 // entries in the queue
  uint32_t cap;
  __device__ __forceinline__ void load(const uint32_t* counters, int q, uint32_t seg_cap) {
    uint32_t s = 0;
#pragma unroll
    for (int g = 0; g < TPT_WF_SEGS; g++) {
      pre[g] = s;
      s += (uint32_t)__builtin_amdgcn_readfirstlane((int)counters[TPT_CNT_IDX(q, g)]);
    }
    n = s;
    cap = seg_cap;
  }
  __device__ __forceinline__ uint32_t slot(uint32_t i) const {
    uint32_t base = 0, off = i;
#pragma unroll
    for (int g = 1; g < TPT_WF_SEGS; g++) {
      if (i >= pre[g]) {
        base = (uint32_t)g * cap;
        off = i - pre[g];
      }
    }
    return base + off;
  }
};

struct WfParams {
  SceneF32 S;
  SmallScene small;
  SceneF64 S64;  // reference-layout scene, for the light self-occlusion decision
  EnvDev env;
  LightsDev lights;
  MatsDev mats;
  CamF32 cam;
  PathState ps;
  int32_t* gstack;  // per-thread overflow stacks (may be null)
  int32_t gstack_cap;
  int32_t width, height;
  int32_t max_bounces, rr_start;
  float inv_w, inv_h;
  uint64_t seed;
  int32_t refill;  // persistent traversal after the first bounce: rays start once fewer than this many lanes of a
                   // wave are tracing (0: one ray per lane)
  int32_t pad;
};

// Path order of a pass of n_pixels pixels and k samples: the pixels in groups of TPT_WF_PIX_GROUP
// (the last one may hold fewer), a group's paths together, sample after sample.  A wave's 64
// camera rays then start in a few pixels and the rays in flight on the chip cover a small part of
// the image, so they meet the same nodes, triangles and materials; sample-major order (path i is
// pixel i mod n_pixels) had the whole image in flight.  Groups of 2 measured best (against
// sample-major order on MI355X: default scene 256^2 x 64 spp 873 -> 759 us, Cornell 512^2 x 256 spp
// 28.5 -> 27.85 ms, 1.31M-triangle mesh 1080p x 32 spp 47.5 -> 44.7 ms, 4096 instances adaptive
// 56.2 -> 53.5 ms; groups of 4 781 us, 27.95, 44.9, 54.2; of 16 787 us, 27.9, 45.6, 55.6; one pixel
// at a time reads the sums uncoalesced: Cornell 28.1).
#define TPT_WF_PIX_GROUP 2
// Path i: pixel `pix` of the pass's pixel set, sample `s` of the samples the pass adds to it.
__host__ __device__ __forceinline__ void path_pixel(uint32_t i, uint32_t n_pixels, uint32_t k, uint32_t* pix,
                                                    uint32_t* s) {
  const uint32_t g = i / (TPT_WF_PIX_GROUP * k), r = i - g * (TPT_WF_PIX_GROUP * k);
  const uint32_t p0 = g * TPT_WF_PIX_GROUP, left = n_pixels - p0;
  if (left >= TPT_WF_PIX_GROUP) {
    *pix = p0 + r % TPT_WF_PIX_GROUP;
    *s = r / TPT_WF_PIX_GROUP;
  } else {
    *pix = p0 + r % left;
    *s = r / left;
  }
}
// First path of pixel `pix` and the stride between its samples' paths.
__host__ __device__ __forceinline__ void path_index(uint32_t pix, uint32_t n_pixels, uint32_t k, uint32_t* first,
                                                    uint32_t* stride) {
  const uint32_t p0 = pix / TPT_WF_PIX_GROUP * TPT_WF_PIX_GROUP, left = n_pixels - p0;
  *first = p0 * k + (pix - p0);
  *stride = left >= TPT_WF_PIX_GROUP ? TPT_WF_PIX_GROUP : left;
}

// The paths of one pass, in the order above.
struct PassArgs {
  uint32_t n_paths;   // pixels * k
  uint32_t n_pixels;  // pixels in this pass
  uint32_t k;         // samples of each pixel
  uint32_t pixel0;    // first pixel (non-adaptive)
  uint32_t s0;        // first sample index (non-adaptive)
  const int32_t* active;  // adaptive: active pixel list (else null)
  const uint32_t* nsamp;  // adaptive: samples taken per pixel
  const int32_t* pix_map;  // image pixel of each domain pixel (null: the domain is the image)
};

// Where the kernels after a bounce's shading tell the host how many paths the next bounce has: a
// word of pinned host memory that receives tag << 32 | paths when such a kernel starts.
struct PathCount {
  uint64_t* seen;  // device address (null: not told)
  uint32_t tag;
  int32_t queue;   // the path queue counted (0 or 1)
};

struct AccumArgs {
  uint32_t n_pixels, pixel0, k;
  double* acc;
  double* acc_w;
  double* acc_sq;
};

struct AdaptiveArgs {
  uint32_t n_active, k, min_spp, max_spp;
  double threshold;
  const int32_t* active_in;
  int32_t* active_out;
  uint32_t* n_active_out;
  uint32_t* nsamp;
  double* welford;  // mean, m2 per pixel
  double* acc;
  double* acc_w;
  double* acc_sq;
};

hipError_t wf_launch_clear_radiance(const WfParams& W, uint32_t n, hipStream_t s);
// gen: the pass's paths, for the first bounce (its kernels generate the camera rays); null after
// ev0 / ev1 (optional): events the dispatch itself records at the kernel's start and end (no
// separate marker packets between kernels)
// count: where a launch after a bounce's shading reports the next bounce's paths (all of them do, the
// first one in time)
hipError_t wf_launch_extend(const WfParams& W, int cur, const PassArgs* gen, const PathCount& count, uint32_t max_n,
                            hipStream_t s, hipEvent_t ev0 = nullptr, hipEvent_t ev1 = nullptr);
// the rest of n paths: gen: the whole paths of a small pass; null: the paths of queue cur, whose
// hits this bounce's extension has stored
hipError_t wf_launch_tail(const WfParams& W, int cur, const PassArgs* gen, uint32_t n, hipStream_t s);
hipError_t wf_launch_shade(const WfParams& W, int cur, const PassArgs* gen, uint32_t max_n, hipStream_t s);
// cur: the queue of paths shaded this bounce; gen: the pass's paths on the first bounce (their
// rays are generated again from their ids), null after
hipError_t wf_launch_light_selfocc(const WfParams& W, int cur, const PassArgs* gen, const PathCount& count,
                                   uint32_t max_n, hipStream_t s);
hipError_t wf_launch_shadow(const WfParams& W, int queue, const PathCount& count, uint32_t max_n, hipStream_t s);
hipError_t wf_launch_accumulate(const WfParams& W, const AccumArgs& A, hipStream_t s);
hipError_t wf_launch_accumulate_adaptive(const WfParams& W, const AdaptiveArgs& A, hipStream_t s);
uint32_t wf_grid_threads(uint32_t n);

// trace_closest entry (k_trace.hip)
// max_blocks > 0 caps the grid (each thread then traces several rays); gstack holds gcap
// overflow entries per thread of the launched grid
hipError_t launch_trace_closest(const SceneF32& S, int64_t n, const float* rays, float* t, int32_t* kind, int32_t* inst,
                                int32_t* prim, int32_t* gstack, int32_t gcap, hipStream_t s, uint32_t max_blocks = 0);
uint32_t trace_grid_threads(int64_t n);  // threads of the default grid for n rays
uint32_t trace_block_threads();          // threads per block

}  // namespace tpt
