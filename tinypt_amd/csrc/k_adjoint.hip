// k_adjoint.hip -- path-replay adjoint of the FP32 render (gradients of a pixel loss with respect
// to material parameters).
//
// Every (pixel, sample) path is regenerated from its seed, seed_for(x, y, s) ^ seed, with the
// same random-number consumption as the forward wavefront kernels, so the adjoint sees exactly
// the paths the forward render summed.  Nothing is stored between paths; passes A and B below
// are one walk for paths short enough to log their BSDF vertices (ADJ_SUMGRAD), two otherwise.
//   Pass A sums, over the path's radiance terms c_k (misses, emitter hits, unoccluded NEE),
//     s_k = x_k o (delta^T J_k), where x_k is the term before the firefly clamp, J_k the clamp's
//     Jacobian (identity when not clamped) and delta = dLoss/dPixel / spp.
//   Pass B walks the path again.  A term's own parameters (BSDF value and MIS weight of its
//     vertex, emitter radiance) are differentiated where the term is formed; a BSDF sample's
//     weight w_j scales every later term, so its parameters receive
//     sum_c (dw_jc/dtheta / w_jc) * (S_total - S_upto_j)_c, the suffix of the pass-A sum.
// Sampling pdfs (BSDF, light selection, env) and Russian-roulette probabilities are held fixed:
// none of these parameters moves a sample, so differentiating the integrand alone gives the
// derivative of the expected image.  Parameters: per material 4 slots laid out like mat_param --
// Lambert / Metal / Subsurface albedo rgb, GGX F0 rgb, Dielectric absorption rgb, DiffuseLight
// emit rgb.
//
// GGX roughness is the exception.  The VNDF sampler of material.rs:327-347 does not draw
// directions with the density its pdf formula (material.rs:283-293) states, and the support
// of the density it does draw from has an edge that moves with alpha, so the expected image
// depends on alpha through the sampler in a way no per-sample derivative captures.  Its
// gradient is therefore taken by replay with common random numbers: every path that meets a
// GGX material is replayed with that material's alpha at +-TPT_ADJ_ALPHA_H and the central
// difference of its loss contribution is added.  The sum over paths is the central difference
// of the whole render's loss with the same seeds, computed in one pass.
#include <string>
#include <vector>

#include "adjoint.h"
#include "tpt_sample32.h"
#include "tpt_selfocc64.h"
#include "wavefront.h"

namespace tpt {

#define TPT_ADJ_BLOCK 256
#define TPT_ADJ_ITEMS 128      // roughness items of a wave at once (at least 64)
#define TPT_ADJ_LDS_GRAD 1024  // per-block gradient slots in LDS (256 materials)
#define TPT_ADJ_ALPHA_H 1e-3  // roughness step of the per-path central difference
#define TPT_ADJ_MAX_GGX 16     // distinct GGX materials per path that receive a roughness gradient

// Replay modes: SUM returns S_total (and lists the path's GGX materials), GRAD accumulates the
// gradients, VALUE returns the path's loss contribution delta . L with one material's roughness
// shifted.  SUMGRAD does SUM and GRAD in one replay: a BSDF vertex's suffix term needs S_total,
// so the vertex's factors and S_upto are logged and the terms added once the path is done --
// possible when a path has at most TPT_ADJ_LOG BSDF vertices (max_bounces <= TPT_ADJ_LOG + 1).
#define ADJ_SUM 0
#define ADJ_GRAD 1
#define ADJ_VALUE 2
#define ADJ_SUMGRAD 3
#define TPT_ADJ_LOG 8

// BSDF vertices of one path whose weight gradient waits for S_total: the term for channel c is
// (S_total - S_upto)_c * num_c / den_c, skipped where den_c = 0.
struct VertexLog {
  int n;
  int mat[TPT_ADJ_LOG];
  f3 num[TPT_ADJ_LOG], den[TPT_ADJ_LOG], s_upto[TPT_ADJ_LOG];
};

struct GgxList {
  int n;
  int mat[TPT_ADJ_MAX_GGX];
  __device__ __forceinline__ void add(int m) {
    for (int i = 0; i < n; i++)
      if (mat[i] == m) return;
    if (n < TPT_ADJ_MAX_GGX) mat[n++] = m;
  }
};

struct AdjParams {
  SceneF32 S;
  SmallScene small;
  SceneF64 S64;  // reference-layout scene, for the light self-occlusion decision
  EnvDev env;
  LightsDev lights;
  MatsDev mats;
  CamF32 cam;
  int32_t* gstack;
  int32_t gcap;
  int32_t width, height, spp, max_bounces, rr_start, n_mats;
  float inv_w, inv_h;
  uint64_t seed;
  uint64_t n_paths;
  const float* dldp;  // w*h*3
  const float* alpha_pm;  // n_mats*2: (float)(alpha + h), (float)(alpha - h)
  double* grad;       // n_mats*4
  uint64_t* stats;    // [0] extension rays, [1] shadow rays, [2] paths
};

// Firefly clamp (math.rs:42-49) and v^T J for its Jacobian.
__device__ __forceinline__ f3 clamp_vjp(f3 x, f3 v) {
  const float m = (float)TPT_FIREFLY_CLAMP;
  float l = luminance(x);
  if (!(l > m && l > 0.f)) return v;
  f3 lam = mk(0.2126f, 0.7152f, 0.0722f);
  float vx = dot(v, x);
  return (m / l) * v - (m * vx / (l * l)) * lam;
}

// d ggx_eval / dF0_c at (n, wo, wi) (material.rs:272-281): (1 - (1 - |wi.m|)^5) D G / denom,
// the same for every channel.
__device__ __forceinline__ float ggx_df_dF0(float s, f3 n, f3 wo, f3 wi) {
  float alpha = fmaxf(s, 1e-3f);
  float ci = dot(n, wo), co = dot(n, wi);
  if (ci <= 0.f || co <= 0.f) return 0.f;
  f3 m = vnorm(wo + wi);
  float ch = fmaxf(dot(n, m), 0.f);
  float D = ggx_distribution(alpha, ch);
  float G = ggx_smith_g1(alpha, ci) * ggx_smith_g1(alpha, co);
  float denom = 4.f * ci * co + 1e-6f;
  float p5 = pow5(1.f - fmaxf(fabsf(dot(wi, m)), 0.f));
  return (1.f - p5) * (D * G / denom);
}

struct GradSink {
  float* lds;  // block slots (or null)
  double* global;
  int n;
  __device__ __forceinline__ void add(int mat, int k, float v) {
    if (v == 0.f || !(v == v)) return;
    int i = 4 * mat + k;
    if (lds && i < TPT_ADJ_LDS_GRAD) atomicAdd(lds + i, v);
    else atomicAdd(global + i, (double)v);
  }
};

__device__ __forceinline__ void add_suffix_terms(GradSink& sink, int mat, f3 num, f3 den, f3 suf) {
  if (den.x != 0.f) sink.add(mat, 0, suf.x * num.x / den.x);
  if (den.y != 0.f) sink.add(mat, 1, suf.y * num.y / den.y);
  if (den.z != 0.f) sink.add(mat, 2, suf.z * num.z / den.z);
}

// One path (see the modes above).  VALUE: material pert_mat's roughness is replaced by
// pert_alpha (the FP32 rounding of the FP64 value +- h, as a material update would upload it).
// The mode is a run-time value, so the kernel holds one inlined copy of the replay: a copy per
// mode took 256 VGPRs plus 620 B of private memory per lane and ran one wave per SIMD; one copy
// runs three waves per SIMD (168 VGPRs, some spilled) and the kernel 2.3x faster.
template <bool ENV_NEE, class Tree, class Stack>
__device__ __forceinline__ f3 replay(const int MODE, const AdjParams& A, const Tree& tree, uint32_t x, uint32_t y, uint32_t s, f3 delta,
                                     f3 S_total, GradSink& sink, GgxList* ggx, VertexLog* log, int pert_mat,
                                     float pert_alpha, const Stack& st, uint32_t* n_ext, uint32_t* n_sh) {
  const bool GRAD = MODE == ADJ_GRAD || MODE == ADJ_SUMGRAD;
  RngF32 rng(seed_for(x, y, s) ^ A.seed);
  f3 o, d;
  camera_ray32(A.cam, x, y, A.inv_w, A.inv_h, rng, &o, &d);
  f3 T = mk(1.f, 1.f, 1.f), S_upto = mk(0.f, 0.f, 0.f);
  float last_pdf = 0.f;
  bool last_nd = false;
  for (int bounce = 0; bounce < A.max_bounces; bounce++) {
    HitF32 h;
    (*n_ext)++;
    if (!trace_f32<false, false>(A.S, tree, o, d, (float)TPT_RAY_EPSILON, 1e30f, &h, st)) {
      // miss (integrator.rs:71-83)
      f3 bg = A.env.black ? mk(0.f, 0.f, 0.f) : (ENV_NEE ? env_lookup32(A.env, d) : sky32(d));
      f3 x0 = had(T, bg);
      float w = 1.f, pe = 0.f;
      if (ENV_NEE && last_nd) {
        pe = env_pdf32(A.env, d);
        w = mis_weight(last_pdf, pe);
      }
      f3 xw = x0 * w;
      if (MODE == ADJ_VALUE) S_upto = S_upto + had(clamp_luminance(xw, (float)TPT_FIREFLY_CLAMP), delta);
      else S_upto = S_upto + had(xw, clamp_vjp(xw, delta));
      break;
    }
    if (bounce >= A.rr_start) {  // integrator.rs:89-95 (probability held fixed)
      float p = fmaxf(fminf(fmaxf(fmaxf(T.x, T.y), T.z), 0.95f), 0.05f);
      if (rng.uni() > p) break;
      T = T / p;
    }
    f3 p, ng;
    int mat;
    hit_geometry32(A.S, h.inst, h.prim, h.t, o, d, &p, &ng, &mat);
    const int kind = A.mats.kind[mat];
    float4 mp = A.mats.p32[mat];
    if (mat == pert_mat) mp.w = pert_alpha;
    const f3 mc = f3of(mp);
    if (kind == TPT_MAT_DIFFUSE_LIGHT) {  // integrator.rs:100-104
      f3 x0 = had(T, mc);
      f3 vj = clamp_vjp(x0, delta);
      if (MODE == ADJ_VALUE) S_upto = S_upto + had(clamp_luminance(x0, (float)TPT_FIREFLY_CLAMP), delta);
      else S_upto = S_upto + had(x0, vj);
      if (GRAD) {
        sink.add(mat, 0, vj.x * T.x);
        sink.add(mat, 1, vj.y * T.y);
        sink.add(mat, 2, vj.z * T.z);
      }
      break;
    }
    if (ggx && kind == TPT_MAT_GGX) ggx->add(mat);
    f3 n = dot(ng, d) < 0.f ? ng : -ng;
    f3 wo = vnorm(-d);
    if (!mat_is_delta(kind)) {
      if (ENV_NEE) {  // nee_environment (integrator.rs:148-172)
        f3 wi, li;
        float pe;
        env_sample32(A.env, rng, &wi, &li, &pe);
        float cs = fmaxf(dot(n, wi), 0.f);
        if (cs > 0.f && pe > 0.f && (li.x != 0.f || li.y != 0.f || li.z != 0.f)) {
          f3 f;
          float pb;
          bsdf_eval(kind, mc, mp.w, wo, wi, n, &f, &pb);
          float w = mis_weight(pe, pb);
          f3 c = had(had(T, f), li) * (cs * w / pe);
          if (c.x != 0.f || c.y != 0.f || c.z != 0.f) {
            HitF32 hs;
            (*n_sh)++;
            if (!trace_f32<true, false>(A.S, tree, p + (float)TPT_RAY_EPSILON * wi, wi, (float)TPT_RAY_EPSILON, 1e30f, &hs, st)) {
              S_upto = S_upto + had(c, delta);
              if (GRAD) {
                f3 base = had(had(T, li), delta) * (cs / pe);  // dc_c/df_c * delta_c / w
                if (kind == TPT_MAT_LAMBERT || kind == TPT_MAT_SUBSURFACE) {
                  sink.add(mat, 0, base.x * w / (float)TPT_PI);
                  sink.add(mat, 1, base.y * w / (float)TPT_PI);
                  sink.add(mat, 2, base.z * w / (float)TPT_PI);
                } else if (kind == TPT_MAT_GGX) {
                  float g = ggx_df_dF0(mp.w, n, wo, wi) * w;
                  sink.add(mat, 0, base.x * g);
                  sink.add(mat, 1, base.y * g);
                  sink.add(mat, 2, base.z * g);
                }
              }
            }
          }
        }
      }
      LightSample32 ls;  // nee_area_light (integrator.rs:178-213)
      if (sample_light32(A.lights, rng, p, &ls)) {
        f3 to_light = ls.pos - p;
        float dist = sqrtf(dot(to_light, to_light));
        if (dist > 1e-6f) {
          f3 wi = to_light / dist;
          float cs = fmaxf(dot(n, wi), 0.f);
          if (cs > 0.f) {
            f3 f;
            float pb;
            bsdf_eval(kind, mc, mp.w, wo, wi, n, &f, &pb);
            float w = mis_weight(ls.pdf, pb);
            f3 c = had(had(T, f), ls.emit) * (cs * w / ls.pdf);
            if ((c.x != 0.f || c.y != 0.f || c.z != 0.f) &&
                !light_self_occluded64(A.S64, A.lights, ls.idx, hit_point64(A.S64, A.S.tri_orig, h.inst, h.prim, o, d, p),
                                       ls.u, ls.v)) {
              float tmax = light_shadow_tmax32(dist);
              HitF32 hs;
              (*n_sh)++;
              if (!trace_f32<true, false>(A.S, tree, p + (float)TPT_RAY_EPSILON * wi, wi, (float)TPT_RAY_EPSILON, tmax, &hs, st)) {
                S_upto = S_upto + had(c, delta);
                if (GRAD) {
                  f3 base = had(had(T, ls.emit), delta) * (cs / ls.pdf);
                  if (kind == TPT_MAT_LAMBERT || kind == TPT_MAT_SUBSURFACE) {
                    sink.add(mat, 0, base.x * w / (float)TPT_PI);
                    sink.add(mat, 1, base.y * w / (float)TPT_PI);
                    sink.add(mat, 2, base.z * w / (float)TPT_PI);
                  } else if (kind == TPT_MAT_GGX) {
                    float g = ggx_df_dF0(mp.w, n, wo, wi) * w;
                    sink.add(mat, 0, base.x * g);
                    sink.add(mat, 1, base.y * g);
                    sink.add(mat, 2, base.z * g);
                  }
                  // emitter radiance of the sampled light
                  f3 e = had(had(T, f), delta) * (cs * w / ls.pdf);
                  sink.add(ls.mat, 0, e.x);
                  sink.add(ls.mat, 1, e.y);
                  sink.add(ls.mat, 2, e.z);
                }
              }
            }
          }
        }
      }
    }
    if (bounce + 1 >= A.max_bounces) break;
    BsdfSample<float> bs;
    if (!bsdf_sample(kind, mc, mp.w, d, p, ng, h.t, rng, &bs)) break;
    if (GRAD) {
      // the sampled weight scales every later term: d log w / d theta times the suffix sum,
      // (S_total - S_upto)_c * num_c / den_c
      f3 num = mk(0.f, 0.f, 0.f), den = num;
      if (kind == TPT_MAT_LAMBERT || kind == TPT_MAT_METAL || kind == TPT_MAT_SUBSURFACE) {
        num = mk(1.f, 1.f, 1.f);  // d log w_c / d albedo_c = 1 / albedo_c
        den = mk(mc.x > 0.f ? mc.x : 0.f, mc.y > 0.f ? mc.y : 0.f, mc.z > 0.f ? mc.z : 0.f);
      } else if (kind == TPT_MAT_GGX) {
        // w_c = F_c D G co / (denom pdf): d log w_c / dF0_c = (1 - (1 - |wi.m|)^5) / F_c
        f3 m = vnorm(wo + bs.d);
        float c = fabsf(dot(bs.d, m));
        f3 F = fresnel_schlick(c, mc);
        float dF = 1.f - pow5(1.f - fmaxf(c, 0.f));
        num = mk(dF, dF, dF);
        den = mk(F.x > 0.f ? F.x : 0.f, F.y > 0.f ? F.y : 0.f, F.z > 0.f ? F.z : 0.f);
      } else if (kind == TPT_MAT_DIELECTRIC && dot(ng, d) >= 0.f) {
        // exiting: weight carries exp(-sigma_c t) (material.rs:111-119)
        float dist = fmaxf(h.t, 0.f);
        num = mk(-dist, -dist, -dist);
        den = mk(1.f, 1.f, 1.f);
      }
      if (den.x != 0.f || den.y != 0.f || den.z != 0.f) {
        if (log) {
          const int j = log->n++;  // fits: a SUMGRAD path has at most TPT_ADJ_LOG BSDF vertices
          log->mat[j] = mat;
          log->num[j] = num;
          log->den[j] = den;
          log->s_upto[j] = S_upto;
        } else {
          add_suffix_terms(sink, mat, num, den, S_total - S_upto);
        }
      }
    }
    T = had(T, bs.weight);
    o = bs.o;
    d = bs.d;
    last_pdf = bs.pdf;
    last_nd = !bs.is_delta;
  }
  return S_upto;
}

struct AdjPath {
  uint32_t x, y, s;
  f3 delta;
};
__device__ __forceinline__ AdjPath adj_path(const AdjParams& A, uint64_t i) {
  AdjPath q;
  const uint32_t npix = (uint32_t)A.width * (uint32_t)A.height;
  const uint32_t pix = (uint32_t)(i % npix);
  q.s = (uint32_t)(i / npix);
  q.x = pix % (uint32_t)A.width;
  q.y = pix / (uint32_t)A.width;
  // the hardware reciprocal by name: written as a division, one build of the kernel rounded it correctly
  // where the others did not, and every gradient at 12 spp moved by an FP32 ulp
  q.delta = mk(A.dldp[3 * pix], A.dldp[3 * pix + 1], A.dldp[3 * pix + 2]) * __builtin_amdgcn_rcpf((float)A.spp);
  return q;
}
// Orders a wave's LDS writes before its lanes' later reads of each other's entries.
__device__ __forceinline__ void wave_lds_sync() {
  __builtin_amdgcn_fence(__ATOMIC_RELEASE, "wavefront");
  __builtin_amdgcn_wave_barrier();
  __builtin_amdgcn_fence(__ATOMIC_ACQUIRE, "wavefront");
}

// The roughness replays of a wave: its lanes' (path, GGX material) items, two neighbouring lanes an
// item, one replaying the path at +h and one at -h (nearly the same path, side by side).  A path
// meets few GGX materials and most meet none, so replaying them lane by lane -- two passes for
// every material of the wave's richest path -- left most lanes idle (12-bounce paths over 20 mesh
// materials, 128^2 x 16 spp: 3.16 -> 2.55 ms).  Each difference is added by the lane whose path it
// is, material by material, so a wave adds its terms in the order of the lane-by-lane form; the
// waves of a block add in FP32 in the order in which they come, as they did, which is what two runs
// differ by (1e-8 to 1e-7 of the gradient's norm).  i: this lane's path; every lane of the wave must
// call it.  Short paths do without: their sums repeat to 1e-9 in part, and adding a wave's roughness
// terms in one burst moves them further than that.
template <bool ENV_NEE, class Tree, class Stack>
__device__ __forceinline__ void replay_items(const AdjParams& A, const Tree& tree, uint64_t i, const GgxList& ggx, uint2* items,
                                             GradSink& sink, const Stack& st, uint32_t* n_ext, uint32_t* n_sh) {
  const uint32_t lane = __lane_id();
  const uint64_t below = (1ull << lane) - 1ull;
  for (int t0 = 0; __any(t0 < ggx.n);) {
    uint32_t k = 0;
    int t1 = t0;
    for (; t1 < TPT_ADJ_MAX_GGX; t1++) {  // the t1-th materials of all lanes, while they fit
      const uint64_t mask = __ballot(t1 < ggx.n);
      const uint32_t c = (uint32_t)__popcll(mask);
      if (c == 0 || k + c > TPT_ADJ_ITEMS) break;
      if (t1 < ggx.n) items[k + (uint32_t)__popcll(mask & below)] = make_uint2(lane, (uint32_t)ggx.mat[t1]);
      k += c;
    }
    wave_lds_sync();
    for (uint32_t b = 0; b < k; b += 32) {
      const uint32_t j = b + (lane >> 1);
      if (j < k) {
        const uint2 it = items[j];
        const AdjPath q = adj_path(A, i - lane + it.x);
        const int m = (int)it.y;
        const f3 v = replay<ENV_NEE>(ADJ_VALUE, A, tree, q.x, q.y, q.s, q.delta, mk(0.f, 0.f, 0.f), sink, nullptr, nullptr, m,
                                     A.alpha_pm[2 * m + (lane & 1)], st, n_ext, n_sh);
        const f3 w = mk(__shfl_xor(v.x, 1), __shfl_xor(v.y, 1), __shfl_xor(v.z, 1));
        if ((lane & 1) == 0) {  // loss term at alpha + h minus the one at alpha - h
          const f3 dv = v - w;
          items[j].x = __float_as_uint((dv.x + dv.y + dv.z) * (float)(0.5 / TPT_ADJ_ALPHA_H));
        }
      }
    }
    wave_lds_sync();
    k = 0;
    for (int t = t0; t < t1; t++) {
      const uint64_t mask = __ballot(t < ggx.n);
      if (t < ggx.n) sink.add(ggx.mat[t], 3, __uint_as_float(items[k + (uint32_t)__popcll(mask & below)].x));
      k += (uint32_t)__popcll(mask);
    }
    wave_lds_sync();
    t0 = t1;
  }
}

// Tree: GlobalTree, or SmallTree for small scenes (tpt_small32.h): replays are bound by the latency of
// a few waves per SIMD, and node loads from LDS shorten it (inverse step of 16 spheres in the Cornell
// box, 256^2 x 16 spp: 5.3 -> 4.75 ms).  OVF: the traversal stack may overflow to global memory;
// ENV_NEE: the environment takes part in next-event estimation; ONE: paths short enough to log (one replay for sums and gradients).
template <class Tree, bool OVF, bool ENV_NEE, bool ONE>
__global__ void __launch_bounds__(TPT_ADJ_BLOCK) __attribute__((amdgpu_waves_per_eu(3))) k_adjoint(AdjParams A) {
  extern __shared__ float4 s_trees[];  // the lanes' stacks, and a small scene's trees
  __shared__ float s_grad[TPT_ADJ_LDS_GRAD];
  __shared__ uint2 s_items[ONE ? 1 : TPT_ADJ_BLOCK / 64 * TPT_ADJ_ITEMS];
  for (int i = threadIdx.x; i < TPT_ADJ_LDS_GRAD; i += blockDim.x) s_grad[i] = 0.f;
  __syncthreads();
  const uint64_t gid = (uint64_t)blockIdx.x * blockDim.x + threadIdx.x;
  LaneStackT<OVF> st;
  const Tree tree = [&] {
    if constexpr (Tree::kWorldOnly) {
      return load_small<TPT_ADJ_BLOCK>(A.S, A.small, s_trees, &st);
    } else {
      st = LaneStackT<OVF>{reinterpret_cast<int32_t*>(s_trees) + threadIdx.x,
                           OVF ? A.gstack + gid * (uint64_t)A.gcap : nullptr, TPT_ADJ_BLOCK, TPT_WF_STACK_ADJ};
      return GlobalTree{A.S};
    }
  }();
  GradSink sink{s_grad, A.grad, A.n_mats};
  uint32_t n_ext = 0, n_sh = 0, n_paths = 0;
  const f3 zero = mk(0.f, 0.f, 0.f);
  if constexpr (ONE) {
    for (uint64_t i = gid; i < A.n_paths; i += (uint64_t)gridDim.x * blockDim.x) {
      const AdjPath q = adj_path(A, i);
      if (q.delta.x == 0.f && q.delta.y == 0.f && q.delta.z == 0.f) continue;
      GgxList ggx;
      ggx.n = 0;
      VertexLog log;
      log.n = 0;
      // pass 0 sums the path's terms (and lists its GGX materials) and takes the gradients; then two
      // passes per GGX material replay the path with its roughness at +h and -h
      f3 dv = zero;
      for (int pass = 0; pass < 1 + 2 * ggx.n; pass++) {
        const int vi = pass - 1;
        const int m = vi >= 0 ? ggx.mat[vi >> 1] : -1;
        const float alpha = vi >= 0 ? A.alpha_pm[2 * m + (vi & 1)] : 0.f;
        const f3 v = replay<ENV_NEE>(pass == 0 ? ADJ_SUMGRAD : ADJ_VALUE, A, tree, q.x, q.y, q.s, q.delta, zero, sink,
                                     pass == 0 ? &ggx : nullptr, pass == 0 ? &log : nullptr, m, alpha, st, &n_ext, &n_sh);
        if (pass == 0) {
          for (int j = 0; j < log.n; j++) add_suffix_terms(sink, log.mat[j], log.num[j], log.den[j], v - log.s_upto[j]);
        } else {  // loss term at alpha + h minus the one at alpha - h
          dv = (vi & 1) ? dv - v : v;
          if (vi & 1) sink.add(m, 3, (dv.x + dv.y + dv.z) * (float)(0.5 / TPT_ADJ_ALPHA_H));
        }
      }
      n_paths++;
    }
  } else {
    for (uint64_t base = (uint64_t)blockIdx.x * blockDim.x; base < A.n_paths; base += (uint64_t)gridDim.x * blockDim.x) {
      const uint64_t i = base + threadIdx.x;
      GgxList ggx;
      ggx.n = 0;
      AdjPath q;
      q.delta = zero;
      if (i < A.n_paths) q = adj_path(A, i);
      if (q.delta.x != 0.f || q.delta.y != 0.f || q.delta.z != 0.f) {
        // pass 0 sums the path's terms (and lists its GGX materials), pass 1 takes the gradients
        f3 S_total = zero;
        for (int pass = 0; pass < 2; pass++)
          S_total = replay<ENV_NEE>(pass == 0 ? ADJ_SUM : ADJ_GRAD, A, tree, q.x, q.y, q.s, q.delta, S_total, sink,
                                    pass == 0 ? &ggx : nullptr, nullptr, -1, 0.f, st, &n_ext, &n_sh);
        n_paths++;
      }
      replay_items<ENV_NEE>(A, tree, i, ggx, s_items + (threadIdx.x >> 6) * TPT_ADJ_ITEMS, sink, st, &n_ext, &n_sh);
    }
  }
  __syncthreads();
  for (int i = threadIdx.x; i < 4 * A.n_mats && i < TPT_ADJ_LDS_GRAD; i += blockDim.x)
    if (s_grad[i] != 0.f) atomicAdd(A.grad + i, (double)s_grad[i]);
  unsigned long long e = n_ext, sh = n_sh, pa = n_paths;
  for (int off = 32; off > 0; off >>= 1) {
    e += (unsigned long long)__shfl_down((long long)e, off);
    sh += (unsigned long long)__shfl_down((long long)sh, off);
    pa += (unsigned long long)__shfl_down((long long)pa, off);
  }
  if (__lane_id() == 0) {
    if (e) atomicAdd((unsigned long long*)&A.stats[0], e);
    if (sh) atomicAdd((unsigned long long*)&A.stats[1], sh);
    if (pa) atomicAdd((unsigned long long*)&A.stats[2], pa);
  }
}

static int adjoint_blocks(uint64_t n_paths) {
  return (int)std::max<uint64_t>(std::min<uint64_t>((n_paths + TPT_ADJ_BLOCK - 1) / TPT_ADJ_BLOCK, 8192), 1);
}

void adjoint_scratch_bytes(const tpt_render_config* cfg, int n_mats, int stack_need, size_t bytes[ADJ_SCRATCH_N]) {
  const size_t npix = (size_t)cfg->width * cfg->height;
  const uint64_t n_paths = (uint64_t)npix * (uint64_t)std::max(cfg->spp, 0);
  const int gcap = stack_need > TPT_WF_STACK_ADJ ? stack_need - TPT_WF_STACK_ADJ : 0;
  bytes[ADJ_SCRATCH_DLDP] = npix * 12;
  bytes[ADJ_SCRATCH_GRAD] = (size_t)std::max(n_mats, 1) * 4 * 8;
  bytes[ADJ_SCRATCH_STATS] = 64;
  bytes[ADJ_SCRATCH_APM] = (size_t)std::max(n_mats, 1) * 2 * 4;
  bytes[ADJ_SCRATCH_GSTACK] = gcap > 0 ? (size_t)adjoint_blocks(n_paths) * TPT_ADJ_BLOCK * gcap * 4 : 0;
}

int adjoint_render(hipStream_t s, const SceneF32& S, const SmallScene& small, const SceneF64& S64, const EnvDev& env, const LightsDev& lights, const MatsDev& mats,
                   const CamF32& cam, const double* mat_param, int stack_need, const tpt_render_config* cfg,
                   const float* d_loss_d_pixel, double* grad_params, tpt_stats* stats, const AdjScratch& scratch,
                   std::string* err) {
  auto fail = [&](int code, const std::string& m) {
    *err = m;
    return code;
  };
  if (cfg->adaptive_enabled) return fail(TPT_ERR_UNSUPPORTED, "the adjoint replays fixed-spp renders only");
  const size_t npix = (size_t)cfg->width * cfg->height;
  const uint64_t n_paths = (uint64_t)npix * (uint64_t)std::max(cfg->spp, 0);
  const int blocks = adjoint_blocks(n_paths);
  const int gcap = stack_need > TPT_WF_STACK_ADJ ? stack_need - TPT_WF_STACK_ADJ : 0;
  std::vector<float> apm(2 * (size_t)std::max(mats.n, 1));
  for (int m = 0; m < mats.n; m++) {
    apm[2 * m] = (float)(mat_param[4 * m + 3] + TPT_ADJ_ALPHA_H);
    apm[2 * m + 1] = (float)(mat_param[4 * m + 3] - TPT_ADJ_ALPHA_H);
  }
  void *d_dldp = scratch.dldp, *d_grad = scratch.grad, *d_stats = scratch.stats, *d_gs = scratch.gstack,
       *d_apm = scratch.apm;
  hipError_t e = hipMemcpyAsync(d_apm, apm.data(), apm.size() * 4, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(d_dldp, d_loss_d_pixel, npix * 12, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemcpyAsync(d_grad, grad_params, (size_t)mats.n * 4 * 8, hipMemcpyHostToDevice, s);
  if (e == hipSuccess) e = hipMemsetAsync(d_stats, 0, 64, s);
  if (e != hipSuccess) return fail(TPT_ERR_DEVICE, std::string("adjoint setup: ") + hipGetErrorString(e));
  AdjParams A{};
  A.S = S;
  A.small = small;
  A.S64 = S64;
  A.env = env;
  A.lights = lights;
  A.mats = mats;
  A.cam = cam;
  A.gstack = (int32_t*)d_gs;
  A.gcap = gcap;
  A.width = cfg->width;
  A.height = cfg->height;
  A.spp = cfg->spp;
  A.max_bounces = cfg->max_bounces;
  A.rr_start = cfg->rr_start;
  A.n_mats = mats.n;
  A.inv_w = (float)(1.0 / (double)cfg->width);
  A.inv_h = (float)(1.0 / (double)cfg->height);
  A.seed = cfg->seed;
  A.n_paths = n_paths;
  A.dldp = (const float*)d_dldp;
  A.alpha_pm = (const float*)d_apm;
  A.grad = (double*)d_grad;
  A.stats = (uint64_t*)d_stats;
  hipEvent_t e0, e1;
  (void)hipEventCreate(&e0);
  (void)hipEventCreate(&e1);
  (void)hipEventRecord(e0, s);
  const bool env_nee = env.kind == TPT_ENV_IMAGE && !env.black;
  const bool one = cfg->max_bounces <= TPT_ADJ_LOG + 1;  // at most max_bounces - 1 BSDF vertices
  const uint32_t lds = small.bytes > 0 ? small_lds(small, TPT_ADJ_BLOCK) : TPT_WF_STACK_ADJ * TPT_ADJ_BLOCK * 4;
  auto launch = [&](auto kernel) { hipLaunchKernelGGL(kernel, dim3(blocks), dim3(TPT_ADJ_BLOCK), lds, s, A); };
  if (n_paths > 0) {
    if (small.bytes > 0) {
      if (env_nee) one ? launch(k_adjoint<SmallTree, false, true, true>) : launch(k_adjoint<SmallTree, false, true, false>);
      else one ? launch(k_adjoint<SmallTree, false, false, true>) : launch(k_adjoint<SmallTree, false, false, false>);
    } else if (gcap > 0) {
      if (env_nee) one ? launch(k_adjoint<GlobalTree, true, true, true>) : launch(k_adjoint<GlobalTree, true, true, false>);
      else one ? launch(k_adjoint<GlobalTree, true, false, true>) : launch(k_adjoint<GlobalTree, true, false, false>);
    } else {
      if (env_nee) one ? launch(k_adjoint<GlobalTree, false, true, true>) : launch(k_adjoint<GlobalTree, false, true, false>);
      else one ? launch(k_adjoint<GlobalTree, false, false, true>) : launch(k_adjoint<GlobalTree, false, false, false>);
    }
  }
  e = hipGetLastError();
  (void)hipEventRecord(e1, s);
  if (e == hipSuccess) e = hipMemcpyAsync(grad_params, d_grad, (size_t)mats.n * 4 * 8, hipMemcpyDeviceToHost, s);
  uint64_t h[8] = {0};
  if (e == hipSuccess) e = hipMemcpyAsync(h, d_stats, 64, hipMemcpyDeviceToHost, s);
  if (e == hipSuccess) e = hipStreamSynchronize(s);
  float ms = 0.f;
  (void)hipEventElapsedTime(&ms, e0, e1);
  (void)hipEventDestroy(e0);
  (void)hipEventDestroy(e1);
  if (e != hipSuccess) return fail(TPT_ERR_DEVICE, std::string("adjoint: ") + hipGetErrorString(e));
  if (stats) {
    stats->paths = h[2];
    stats->rays_extension = h[0];
    stats->rays_shadow = h[1];
    stats->elapsed_ms = ms;
    stats->trace_kernel_ms = ms;
    stats->trace_launches = 1;
    stats->trace_rays = h[0] + h[1];
    stats->light_samples = 0;
    stats->light_self_occluded = 0;
  }
  return TPT_OK;
}

}  // namespace tpt
