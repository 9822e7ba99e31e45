// k_plain64.hip -- the plain FP64 GPU form: the reference's per-pixel random stream across all
// samples (render.rs:142), its trees and its f64 arithmetic without FMA contraction (this file is
// compiled with -ffp-contract=off), one pixel per lane or per four lanes.  It restates
// render.rs:137-191, integrator.rs, world.rs, bvh.rs, geometry.rs, env.rs and material.rs on
// the device and is the baseline the FP32 wavefront is measured against.  Work that cannot change
// a sum is left out: instances a ray cannot hit, second tests of a node that can only repeat the
// first, shadow rays whose contribution is zero.
//
// What bounds it: divergent lanes (20% of them active) and latency at two waves per SIMD; VALUs 21%
// busy.  On MI355X: Cornell box 256^2 x 16 spp 11.4 -> 6.1 ms (every ray taken into all eight
// instances, private stack, one bounce of all lanes until the longest path of a sample ended,
// before), 1024^2 x 4 spp 37 -> 10.4 ms, 82k-triangle mesh 240x135 x 8 spp 19.8 -> 6.9 ms, 1920x1080
// x 1 spp 22 -> 11 ms, 64 instances 240x135 x 8 spp 75 -> 13 ms.
//
// Samples can be split over launches: the per-pixel RNG state, sums and Welford state persist
// in device buffers between chunks, so a chunked render equals an unchunked one.
#include "plain64.h"
#include "tpt_bsdf.h"

namespace tpt {

typedef vec3<double> d3;

// A surface hit, as World::hit returns it.
struct Hit64 {
  double t;
  d3 p, n;
  int mat;
};

// ---------------------------------------------------------------- geometry.rs
// Distance of the sphere along the ray; the hit point and normal follow for the closest hit only.
__device__ __forceinline__ bool sphere_hit(const double* s, d3 o, d3 d, double tmin, double tmax, double* t_out) {
  d3 c = ld3(s);
  double r = s[3];
  d3 oc = o - c;
  double a = dot(d, d);
  double b = dot(oc, d);
  double cc = dot(oc, oc) - r * r;
  double disc = b * b - a * cc;
  if (disc <= 0.0) return false;
  double sd = sqrt(disc);
  double t = (-b - sd) / a;
  if (t < tmin || t > tmax) {
    t = (-b + sd) / a;
    if (t < tmin || t > tmax) return false;
  }
  *t_out = t;
  return true;
}
// vertices_at(time) of a static triangle (geometry.rs:212-218)
__device__ __forceinline__ void tri_verts(const double* v, double time, d3* v0, d3* v1, d3* v2) {
  *v0 = ld3(v) * (1.0 - time) + ld3(v) * time;
  *v1 = ld3(v + 3) * (1.0 - time) + ld3(v + 3) * time;
  *v2 = ld3(v + 6) * (1.0 - time) + ld3(v + 6) * time;
}
__device__ __forceinline__ bool tri_hit(const double* v, d3 o, d3 d, double time, double tmin, double tmax, double* t_out) {
  d3 v0, v1, v2;  // then Moller-Trumbore
  tri_verts(v, time, &v0, &v1, &v2);
  d3 e1 = v1 - v0, e2 = v2 - v0;
  d3 pvec = cross(d, e2);
  double det = dot(e1, pvec);
  if (fabs(det) < 1e-10) return false;
  double inv_det = 1.0 / det;
  d3 tvec = o - v0;
  double u = dot(tvec, pvec) * inv_det;
  if (u < 0.0 || u > 1.0) return false;
  d3 qvec = cross(tvec, e1);
  double vv = dot(d, qvec) * inv_det;
  if (vv < 0.0 || u + vv > 1.0) return false;
  double th = dot(e2, qvec) * inv_det;
  if (th < tmin || th > tmax) return false;
  *t_out = th;
  return true;
}
// Aabb::hit_range: entry distance t0; false when the slabs leave no interval.  (The reference
// returns after the first axis that leaves none; later axes only narrow the interval.)
__device__ __forceinline__ bool aabb_range(const double* b, d3 o, d3 inv, double tmin, double tmax, double* t0) {
  double t0x = (b[0] - o.x) * inv.x, t1x = (b[3] - o.x) * inv.x;
  double t0y = (b[1] - o.y) * inv.y, t1y = (b[4] - o.y) * inv.y;
  double t0z = (b[2] - o.z) * inv.z, t1z = (b[5] - o.z) * inv.z;
  tmin = fmax(tmin, fmin(t0x, t1x));
  tmax = fmin(tmax, fmax(t0x, t1x));
  tmin = fmax(tmin, fmin(t0y, t1y));
  tmax = fmin(tmax, fmax(t0y, t1y));
  tmin = fmax(tmin, fmin(t0z, t1z));
  tmax = fmin(tmax, fmax(t0z, t1z));
  *t0 = tmin;
  return !(tmax <= tmin);
}

// With G = 4 a pixel has four neighbouring lanes (a quad), all with the same state and control
// flow; a value crosses the quad by quad permutations.
template <int CTRL>
__device__ __forceinline__ int quad_get(int v) {
  return __builtin_amdgcn_update_dpp(0, v, CTRL, 0xf, 0xf, true);
}
template <int CTRL>
__device__ __forceinline__ double quad_get(double v) {
  return __hiloint2double(quad_get<CTRL>(__double2hiint(v)), quad_get<CTRL>(__double2loint(v)));
}
// The closest of the quad's triangle hits (slot k, -1: none); of equal distances the last slot's, as
// the reference's loop over a leaf keeps the last.
template <int CTRL>
__device__ __forceinline__ void quad_closest(double& th, int& k, int& tri) {
  const double t2 = quad_get<CTRL>(th);
  const int k2 = quad_get<CTRL>(k), tri2 = quad_get<CTRL>(tri);
  if (k2 >= 0 && (k < 0 || t2 < th || (t2 == th && k2 > k))) {
    th = t2;
    k = k2;
    tri = tri2;
  }
}

// ---------------------------------------------------------------- bvh.rs:248-351
// Traversal stack: what a far child is (inner node, or the range of a leaf) and its entry
// distance.  The first TPT_PLAIN_LDS entries of a lane are in LDS, the rest (the reference's 64;
// the host rejects trees deeper than 63 levels for this form, so the heap spill path of the
// reference is never needed) in private memory.
#define TPT_PLAIN_LDS 8
struct PlainStack {
  double* t_lds;  // this lane's columns
  int2* n_lds;
  double t[64 - TPT_PLAIN_LDS];
  int2 n[64 - TPT_PLAIN_LDS];
  __device__ __forceinline__ void put(int i, int2 node, double t0) {
    if (i < TPT_PLAIN_LDS) {
      t_lds[i * TPT_PLAIN_BLOCK] = t0;
      n_lds[i * TPT_PLAIN_BLOCK] = node;
    } else {
      t[i - TPT_PLAIN_LDS] = t0;
      n[i - TPT_PLAIN_LDS] = node;
    }
  }
  __device__ __forceinline__ double entry(int i) const {
    return i < TPT_PLAIN_LDS ? t_lds[i * TPT_PLAIN_BLOCK] : t[i - TPT_PLAIN_LDS];
  }
  __device__ __forceinline__ int2 node(int i) const {
    return i < TPT_PLAIN_LDS ? n_lds[i * TPT_PLAIN_BLOCK] : n[i - TPT_PLAIN_LDS];
  }
};

// Bvh::hit over PlainNode: the reference's visits in the reference's order.  A node is tested
// when its parent is visited and (for the reference) once more when it is popped; only tmax can
// have changed in between, so the second test is tmax against the entry distance, and none for
// the near child, which is visited at once.
template <int G>
__device__ __forceinline__ bool bvh_hit(const Plain64Params& P, const MeshDev& M, const PlainMesh& R, d3 o, d3 d,
                                        double time, double tmin, double tmax, PlainStack& st, double* t_hit,
                                        int* tri_hit_out) {
  if (R.root == TPT_PLAIN_NONE) return false;
  const PlainNode* nodes = P.nodes + R.node_off;
  const int32_t* idx = P.S.indices + M.idx_off;
  d3 inv = mk(1.0 / d.x, 1.0 / d.y, 1.0 / d.z);
  int sp = 0;
  bool found = false;
  double t0;
  if (!aabb_range(R.box, o, inv, tmin, tmax, &t0)) return false;
  // x >= 0: inner node x; x < 0: leaf, indices y .. y - x - 1
  int2 cur = R.root == TPT_PLAIN_LEAF ? make_int2(-(int)R.count, (int)R.start) : make_int2(R.root, 0);
  if (R.root == TPT_PLAIN_LEAF && R.count == 0) return false;
  bool more = true;
  auto pop = [&]() {
    do {
      if (sp == 0) {
        more = false;
        return;
      }
      sp--;
    } while (tmax <= st.entry(sp));
    cur = st.node(sp);
  };
  while (more) {
    while (more && cur.x >= 0) {
      const PlainNode& n = nodes[cur.x];
      double e[2] = {0.0, 0.0};
      bool in[2];
      int2 kid[2];
#pragma unroll
      for (int k = 0; k < 2; k++) {
        in[k] = aabb_range(n.b[k], o, inv, tmin, tmax, &e[k]) && n.child[k] != TPT_PLAIN_NONE &&
                !(n.child[k] == TPT_PLAIN_LEAF && n.count[k] == 0);
        kid[k] = n.child[k] >= 0 ? make_int2(n.child[k], 0) : make_int2(-(int)n.count[k], (int)n.start[k]);
      }
      if (in[0] && in[1]) {
        const bool a_first = e[0] <= e[1];
        st.put(sp++, a_first ? kid[1] : kid[0], a_first ? e[1] : e[0]);
        cur = a_first ? kid[0] : kid[1];
      } else if (in[0] || in[1]) {
        cur = in[0] ? kid[0] : kid[1];
      } else {
        pop();
      }
    }
    if (!more) break;
    for (int k0 = cur.y; k0 < cur.y - cur.x; k0 += G) {
      int k = k0 + (G > 1 ? (int)(threadIdx.x % G) : 0), ti = 0;
      double th = 0.0;
      if (k < cur.y - cur.x) {
        ti = idx[k];
        if (!tri_hit(P.S.tris + 9 * (size_t)(M.tri_off + ti), o, d, time, tmin, tmax, &th)) k = -1;
      } else {
        k = -1;
      }
      if constexpr (G == 4) {
        quad_closest<0xB1>(th, k, ti);  // lanes 1, 0, 3, 2
        quad_closest<0x4E>(th, k, ti);  // lanes 2, 3, 0, 1
      }
      if (k >= 0) {
        tmax = th;
        *tri_hit_out = ti;
        found = true;
      }
    }
    pop();
  }
  *t_hit = tmax;
  return found;
}

__device__ __forceinline__ d3 mat_vec(const double* m, d3 v) {
  return mk(m[0] * v.x + m[1] * v.y + m[2] * v.z, m[3] * v.x + m[4] * v.y + m[5] * v.z, m[6] * v.x + m[7] * v.y + m[8] * v.z);
}

// ---------------------------------------------------------------- world.rs:81-121
// The reference takes the ray into every instance.  Here an instance whose world box the ray
// misses, or enters beyond the closest hit so far, is skipped by an FP32 slab test: the box is
// grown by `slack`, a multiple of the FP32 rounding of the box, origin and products, so that no
// instance the reference could take a hit from is skipped.  Inside an instance the search stops
// at the closest hit so far (with the same slack) instead of at 1e30: a farther hit would be
// dropped by t_world < closest.  any: whether there is a hit at all (shadow rays), so the first
// instance or sphere with one decides.
template <int G>
__device__ __forceinline__ bool world_hit(const Plain64Params& P, d3 o, d3 d, double time, double tmin, double tmax,
                                          bool any, PlainStack& st, Hit64* best) {
  const SceneF64& S = P.S;
  double closest = tmax;
  int hit_inst = -1, hit_tri = -1, hit_sphere = -1;
  d3 hit_p = mk(0.0, 0.0, 0.0);
  const float ox = (float)o.x, oy = (float)o.y, oz = (float)o.z;
  const float ix = __builtin_amdgcn_rcpf((float)d.x), iy = __builtin_amdgcn_rcpf((float)d.y),
              iz = __builtin_amdgcn_rcpf((float)d.z);
  const float o_max = fmaxf(fmaxf(fabsf(ox), fabsf(oy)), fabsf(oz)) + 1.f;
  for (int ii = 0;; ii++) {
    // this lane's next instance: the cheap test alone runs over the ones it skips, so that the
    // lanes of a wave walk their trees together, whichever instances these are
    float slack = 0.f;
    for (; ii < S.n_inst; ii++) {
      const float* b = P.inst_box + 6 * ii;
      slack = 2e-6f * (o_max + fmaxf(fmaxf(fmaxf(fabsf(b[0]), fabsf(b[1])), fmaxf(fabsf(b[2]), fabsf(b[3]))),
                                                 fmaxf(fabsf(b[4]), fabsf(b[5]))));
      const float x0 = (b[0] - slack - ox) * ix, x1 = (b[3] + slack - ox) * ix;
      const float y0 = (b[1] - slack - oy) * iy, y1 = (b[4] + slack - oy) * iy;
      const float z0 = (b[2] - slack - oz) * iz, z1 = (b[5] + slack - oz) * iz;
      const float in = fmaxf(fmaxf(fminf(x0, x1), fminf(y0, y1)), fminf(z0, z1));
      const float out = fminf(fminf(fmaxf(x0, x1), fmaxf(y0, y1)), fmaxf(z0, z1));
      if (!(slack < 1e30f && (in > out || out < 0.f || in > (float)closest * 1.000002f + slack))) break;
    }
    if (ii >= S.n_inst) break;
    const InstF64& I = S.inst[ii];
    if (I.mesh < 0 || I.mesh >= S.n_meshes) continue;
    d3 o_obj = mat_vec(I.a_inv, o - ld3(I.t));
    d3 d_obj = mat_vec(I.a_inv, d);
    const double l = fmax(vlen(d_obj), 1e-30);  // vnorm (math.rs:69-72)
    d_obj = d_obj / l;
    double th;
    int tri;
    if (bvh_hit<G>(P, S.meshes[I.mesh], P.meshes[I.mesh], o_obj, d_obj, time, tmin,
                fmin((closest * (1.0 + 1e-6) + (double)slack) * l, 1e30), st, &th, &tri)) {
      d3 p_world = mat_vec(I.a, o_obj + d_obj * th) + ld3(I.t);
      double t_world = dot(p_world - o, d);
      if (t_world > tmin && t_world < closest) {
        if (any) return true;
        closest = t_world;
        hit_inst = ii;
        hit_tri = tri;
        hit_p = p_world;
      }
    }
  }
  for (int s = 0; s < S.n_spheres; s++) {
    double t;
    if (sphere_hit(S.sph + 4 * s, o, d, tmin, closest, &t)) {
      if (any) return true;
      closest = t;
      hit_sphere = s;
    }
  }
  if (any) return false;
  best->t = closest;
  if (hit_sphere >= 0) {
    const double* s = S.sph + 4 * hit_sphere;
    best->p = o + d * closest;
    best->n = (best->p - ld3(s)) / s[3];
    best->mat = S.sph_mat[hit_sphere];
    return true;
  }
  if (hit_inst < 0) return false;
  const InstF64& I = S.inst[hit_inst];
  const MeshDev& M = S.meshes[I.mesh];
  d3 v0, v1, v2;
  tri_verts(S.tris + 9 * (size_t)(M.tri_off + hit_tri), time, &v0, &v1, &v2);
  best->p = hit_p;
  best->n = vnorm(mat_vec(I.nrm, vnorm(cross(v1 - v0, v2 - v0))));
  best->mat = I.mat_override >= 0 ? I.mat_override : S.tri_mat[M.tri_off + hit_tri];
  return true;
}

// ---------------------------------------------------------------- env.rs
__device__ __forceinline__ void dir_uv64(d3 dir, double* u, double* v, double* theta) {
  d3 d = vnorm(dir);
  double th = acos(fmin(fmax(d.y, -1.0), 1.0));
  double phi = atan2(d.z, d.x);
  if (phi < 0.0) phi += TPT_TAU;
  *u = phi / TPT_TAU;
  *v = th / TPT_PI;
  *theta = th;
}
__device__ __forceinline__ size_t as_usize(double v) { return v > 0.0 ? (size_t)v : 0; }
__device__ d3 env_lookup64(const EnvDev& E, d3 dir) {  // env.rs:92-121
  double u, v, th;
  dir_uv64(dir, &u, &v, &th);
  double x = u * (double)E.w;
  double y = v * ((double)E.h - 1.0);
  size_t x0 = as_usize(floor(x)) % (size_t)E.w;
  size_t x1 = (x0 + 1) % (size_t)E.w;
  size_t y0 = as_usize(floor(fmin(fmax(y, 0.0), (double)(E.h - 1))));
  size_t y1 = y0 + 1 < (size_t)(E.h - 1) ? y0 + 1 : (size_t)(E.h - 1);
  double fx = x - floor(x), fy = y - floor(y);
  d3 c00 = ld3(E.rgb64 + 3 * (y0 * E.w + x0)), c10 = ld3(E.rgb64 + 3 * (y0 * E.w + x1));
  d3 c01 = ld3(E.rgb64 + 3 * (y1 * E.w + x0)), c11 = ld3(E.rgb64 + 3 * (y1 * E.w + x1));
  d3 c0 = c00 * (1.0 - fx) + c10 * fx;
  d3 c1 = c01 * (1.0 - fx) + c11 * fx;
  return c0 * (1.0 - fy) + c1 * fy;
}
__device__ double env_pdf64(const EnvDev& E, d3 dir) {  // env.rs:156-182
  if (E.total <= 0.0) return 1.0 / (4.0 * TPT_PI);
  double u, v, theta;
  dir_uv64(dir, &u, &v, &theta);
  double fxv = floor(u * (double)E.w), fyv = floor(v * (double)E.h);
  if (fxv < 0.0) fxv = 0.0;
  if (fxv > (double)(E.w - 1)) fxv = (double)(E.w - 1);
  if (fyv < 0.0) fyv = 0.0;
  if (fyv > (double)(E.h - 1)) fyv = (double)(E.h - 1);
  size_t x = as_usize(fxv), y = as_usize(fyv);
  double theta0 = TPT_PI * (double)y / (double)E.h;
  double theta1 = TPT_PI * (double)(y + 1) / (double)E.h;
  double sin_theta = fmax(sin(theta), 1e-6);
  double row_weight = fmax(cos(theta0) - cos(theta1), 0.0);
  double l = fmax(luminance(ld3(E.rgb64 + 3 * (y * E.w + x))), 0.0);
  double weight = l * row_weight;
  if (weight <= 0.0) return 0.0;
  double pdf_uv = (weight / E.total) * (double)E.w * (double)E.h;
  return pdf_uv / (2.0 * TPT_PI * TPT_PI * sin_theta);
}
__device__ void env_sample64(const EnvDev& E, RngF64& rng, d3* dir, d3* li, double* pdf) {  // env.rs:124-152, 200-210
  bool uniform = E.total <= 0.0;
  int y = 0;
  double row_sum = 0.0;
  if (!uniform) {
    double r0 = rng.uni() * E.total;
    y = min(cdf_search(E.row_cdf, E.h + 1, r0), E.h - 1);
    row_sum = fmax(E.row_cdf[y + 1] - E.row_cdf[y], 0.0);
    if (row_sum <= 0.0) uniform = true;
  }
  if (uniform) {
    double u = rng.uni(), v = rng.uni();
    double z = 1.0 - 2.0 * u;
    double r = sqrt(fmax(1.0 - z * z, 0.0));
    double phi = TPT_TAU * v;
    *dir = mk(r * cos(phi), z, r * sin(phi));
    *li = E.black ? mk(0.0, 0.0, 0.0) : env_lookup64(E, *dir);
    *pdf = 1.0 / (4.0 * TPT_PI);
    return;
  }
  double r1 = rng.uni() * row_sum;
  int x = min(cdf_search(E.col_cdf + (size_t)y * (E.w + 1), E.w + 1, r1), E.w - 1);
  double u = ((double)x + rng.uni()) / (double)E.w;
  double v = ((double)y + rng.uni()) / (double)E.h;
  double theta = TPT_PI * v, phi = TPT_TAU * u;
  double st = sin(theta);
  *dir = mk(cos(phi) * st, cos(theta), sin(phi) * st);
  *li = env_lookup64(E, *dir);
  *pdf = env_pdf64(E, *dir);
}

// ---------------------------------------------------------------- lights (world.rs:171-272)
__device__ __forceinline__ void tri_world_verts(const SceneF64& S, const LightF64& L, double time, d3* a, d3* b, d3* c) {
  const InstF64& I = S.inst[L.inst];
  const double* v = S.tris + 9 * (size_t)(S.meshes[L.mesh].tri_off + L.tri);
  d3 v0 = ld3(v) * (1.0 - time) + ld3(v) * time;
  d3 v1 = ld3(v + 3) * (1.0 - time) + ld3(v + 3) * time;
  d3 v2 = ld3(v + 6) * (1.0 - time) + ld3(v + 6) * time;
  *a = mat_vec(I.a, v0) + ld3(I.t);
  *b = mat_vec(I.a, v1) + ld3(I.t);
  *c = mat_vec(I.a, v2) + ld3(I.t);
}
struct LightSample64 {
  d3 pos, nrm, emit;
  double pdf;
};
__device__ bool sample_light64(const SceneF64& S, const LightsDev& Ls, RngF64& rng, double time, d3 p, LightSample64* out) {
  if (Ls.total <= 0.0 || Ls.n == 0) return false;
  double r = rng.uni() * Ls.total;
  int idx = min(cdf_search(Ls.cdf64, Ls.n, r), Ls.n - 1);
  const LightF64& L = Ls.l64[idx];
  double pdf_select = L.weight / Ls.total;
  d3 pos, nrm;
  double area;
  if (L.kind == 0) {
    const double* s = S.sph + 4 * L.idx;
    double u = rng.uni(), v = rng.uni();
    double z = 1.0 - 2.0 * u;
    double rr = sqrt(fmax(1.0 - z * z, 0.0));
    double phi = TPT_TAU * v;
    d3 dir = mk(rr * cos(phi), z, rr * sin(phi));
    pos = ld3(s) + dir * s[3];
    nrm = dir;
    area = 4.0 * TPT_PI * s[3] * s[3];
  } else {
    d3 a, b, c;
    tri_world_verts(S, L, time, &a, &b, &c);
    double u = rng.uni(), v = rng.uni();
    double su = sqrt(u);
    double b0 = 1.0 - su, b1 = v * su, b2 = 1.0 - b0 - b1;
    pos = a * b0 + b * b1 + c * b2;
    d3 n = cross(b - a, c - a);
    area = 0.5 * vlen(n);
    nrm = area > 0.0 ? n / (2.0 * area) : mk(0.0, 1.0, 0.0);
  }
  if (area <= 0.0) return false;
  d3 to_light = pos - p;
  double dist2 = dot(to_light, to_light);
  if (dist2 <= 1e-12) return false;
  double dist = sqrt(dist2);
  d3 wi = to_light / dist;
  double cos_light = fmax(dot(nrm, -wi), 0.0);
  if (cos_light <= 0.0) return false;
  double pdf_area = 1.0 / area;
  double pdf_omega = pdf_area * dist2 / cos_light;
  double pdf = pdf_select * pdf_omega;
  if (pdf <= 0.0) return false;
  out->pos = pos;
  out->nrm = nrm;
  out->emit = mk(L.emit[0], L.emit[1], L.emit[2]);
  out->pdf = pdf;
  return true;
}

// ---------------------------------------------------------------- integrator.rs:53-213
struct Count64 {
  uint32_t ext, shadow;
};
// A path on its way.  radiance() is cut at its rays: a vertex's shadow rays and the next
// extension ray wait here, and the lanes of a wave trace theirs side by side through one copy of the
// traversal.  (No random draw depends on a shadow ray's result, so the draws keep the reference's
// order.)
struct Path64 {
  d3 ro, rd, acc, beta;  // the extension ray
  double time, last_bsdf_pdf;
  int bounce;
  bool last_non_delta, alive;  // alive: the extension ray is to be traced
  bool env, light;             // shadow rays to be traced first
  double* sh;  // they wait in LDS, in this lane's column: origin, direction, contribution, tmax
  __device__ __forceinline__ void put_shadow(int which, d3 o, d3 d, d3 c, double tmax) {
    double* p = sh + which * 10 * TPT_PLAIN_BLOCK;
    const double v[10] = {o.x, o.y, o.z, d.x, d.y, d.z, c.x, c.y, c.z, tmax};
#pragma unroll
    for (int k = 0; k < 10; k++) p[k * TPT_PLAIN_BLOCK] = v[k];
  }
  __device__ __forceinline__ d3 shadow3(int which, int k) const {
    const double* p = sh + (which * 10 + k) * TPT_PLAIN_BLOCK;
    return mk(p[0], p[TPT_PLAIN_BLOCK], p[2 * TPT_PLAIN_BLOCK]);
  }
};

// Whether a contribution changes the sum it is added to (a zero need not wait for its shadow ray,
// which is counted all the same).
__device__ __forceinline__ bool adds(d3 c) { return !(c.x == 0.0 && c.y == 0.0 && c.z == 0.0); }

// The path at its extension ray's hit, or miss (integrator.rs:53-213).
__device__ __forceinline__ void vertex64(const Plain64Params& P, Path64& q, bool found, const Hit64& hit, RngF64& rng,
                                         Count64* cnt) {
  const SceneF64& S = P.S;
  const bool has_env = P.env.kind == TPT_ENV_IMAGE;
  const d3 rd = q.rd;
  q.alive = false;
  if (!found) {
    if (P.env.black) return;  // adds zero
    d3 bg;
    if (has_env) bg = env_lookup64(P.env, rd);
    else {
      double t = 0.5 * (rd.y + 1.0);
      bg = (1.0 - t) * mk(0.9, 0.95, 1.0) + t * mk(0.6, 0.75, 1.0);
    }
    d3 contrib = had(q.beta, bg);
    if (has_env && q.last_non_delta) contrib = contrib * mis_weight(q.last_bsdf_pdf, env_pdf64(P.env, rd));
    q.acc = q.acc + clamp_luminance(contrib, TPT_FIREFLY_CLAMP);
    return;
  }
  if (q.bounce >= P.rr_start) {
    double p = fmax(fmin(fmax(fmax(q.beta.x, q.beta.y), q.beta.z), 0.95), 0.05);
    if (rng.uni() > p) return;
    q.beta = q.beta / p;
  }
  const int kind = P.mats.kind[hit.mat];
  const double* mp = P.mats.p64 + 4 * hit.mat;
  const d3 mc = ld3(mp);
  if (kind == TPT_MAT_DIFFUSE_LIGHT) {
    q.acc = q.acc + clamp_luminance(had(q.beta, mc), TPT_FIREFLY_CLAMP);
    return;
  }
  d3 n = dot(hit.n, rd) < 0.0 ? hit.n : -hit.n;
  if (!mat_is_delta(kind)) {
    if (has_env) {  // nee_environment
      d3 wi, li;
      double pdf_env;
      env_sample64(P.env, rng, &wi, &li, &pdf_env);
      double cs = fmax(dot(n, wi), 0.0);
      if (cs > 0.0 && pdf_env > 0.0) {
        cnt->shadow++;
        d3 f;
        double pdf_b;
        bsdf_eval(kind, mc, mp[3], vnorm(-rd), wi, n, &f, &pdf_b);
        double w = mis_weight(pdf_env, pdf_b);
        const d3 c = had(had(q.beta, f), li) * (cs * w / pdf_env);
        q.env = adds(c);
        if (q.env) q.put_shadow(0, hit.p + TPT_RAY_EPSILON * wi, wi, c, 1e30);
      }
    }
    LightSample64 ls;  // nee_area_light
    if (sample_light64(S, P.lights, rng, q.time, hit.p, &ls)) {
      d3 to_light = ls.pos - hit.p;
      double dist2 = dot(to_light, to_light);
      double dist = sqrt(dist2);
      if (dist > 1e-6) {
        d3 wi = to_light / dist;
        double cs = fmax(dot(n, wi), 0.0);
        if (cs > 0.0) {
          cnt->shadow++;
          d3 f;
          double pdf_b;
          bsdf_eval(kind, mc, mp[3], vnorm(-rd), wi, n, &f, &pdf_b);
          const d3 c = had(had(q.beta, f), ls.emit) * (cs * mis_weight(ls.pdf, pdf_b) / ls.pdf);
          q.light = ls.pdf > 0.0 && adds(c);
          if (q.light)
            q.put_shadow(1, hit.p + TPT_RAY_EPSILON * wi, wi, c, fmax(dist - TPT_RAY_EPSILON, TPT_RAY_EPSILON));
        }
      }
    }
  }
  BsdfSample<double> bs;
  if (!bsdf_sample(kind, mc, mp[3], rd, hit.p, hit.n, hit.t, rng, &bs)) return;
  q.last_bsdf_pdf = bs.pdf;
  q.last_non_delta = !bs.is_delta;
  q.beta = had(q.beta, bs.weight);
  q.ro = bs.o;
  q.rd = bs.d;
  q.alive = ++q.bounce < P.max_bounces;
}

// ---------------------------------------------------------------- render.rs:137-191
// A pixel's samples share one random stream, so a lane works through its pixel's samples in
// order, taking the next sample as soon as a path ends.  G lanes per pixel (1 or 4), P.shape.lanes lanes of
// the wave in use (a multiple of G).
template <int G>
__global__ void __launch_bounds__(TPT_PLAIN_BLOCK) __attribute__((amdgpu_waves_per_eu(2))) k_plain64(Plain64Params P) {
  __shared__ double s_t[TPT_PLAIN_LDS * TPT_PLAIN_BLOCK];
  __shared__ int2 s_n[TPT_PLAIN_LDS * TPT_PLAIN_BLOCK];
  __shared__ double s_sh[20 * TPT_PLAIN_BLOCK];
  // domain pixel: indexes the sums and state
  const int pix = (int)(((int64_t)blockIdx.x * P.shape.lanes + threadIdx.x) / G);
  Count64 cnt{0, 0};
  uint32_t paths = 0;
  if ((int)threadIdx.x < P.shape.lanes && pix < P.n_pix && !P.done[pix]) {
    PlainStack st;
    st.t_lds = s_t + threadIdx.x;
    st.n_lds = s_n + threadIdx.x;
    const int img = P.pix_map ? P.pix_map[pix] : pix;
    const int x = img % P.width, y = img / P.width;
    RngF64 rng(1);
    rng.p.state = P.s_begin == 0 ? Pcg32(seed_for((uint32_t)x, (uint32_t)y, 0) ^ P.seed).state : P.rng[pix];
    const bool writes = G == 1 || threadIdx.x % G == 0;  // one lane of a pixel's writes and counts
    uint32_t n = P.s_begin == 0 ? 0u : P.nsamp[pix];
    double mean = P.s_begin == 0 ? 0.0 : P.welford[2 * pix], m2 = P.s_begin == 0 ? 0.0 : P.welford[2 * pix + 1];
    bool done = false;
    const CameraF64& C = P.cam;
    const uint32_t max_spp = (uint32_t)max(P.spp, 1);
    const uint32_t min_spp = min((uint32_t)max(P.min_spp, 1), max_spp);
    Path64 q;
    q.alive = q.env = q.light = false;
    q.sh = s_sh + threadIdx.x;
    for (int s = P.s_begin;;) {
      if (!(q.alive || q.env || q.light)) {
        if (s >= P.s_end || done) break;
        double jx = rng.uni(), jy = rng.uni();
        double sx = ((double)x + jx) * P.inv_w * 2.0 - 1.0;
        double sy = 1.0 - ((double)y + jy) * P.inv_h * 2.0;
        // Camera::ray (ray.rs:91-108)
        d3 dir_base = vnorm(-ld3(C.w) + (sx * C.half_w) * ld3(C.u) + (sy * C.half_h) * ld3(C.v));
        d3 lens = mk(0.0, 0.0, 0.0);
        if (C.lens_radius > 0.0) {
          double dx = 0.0, dy = 0.0;
          for (int tries = 0; tries < 1024; tries++) {
            double a = 2.0 * rng.uni() - 1.0, b = 2.0 * rng.uni() - 1.0;
            if (a * a + b * b < 1.0) { dx = a; dy = b; break; }
          }
          lens = ld3(C.u) * (dx * C.lens_radius) + ld3(C.v) * (dy * C.lens_radius);
        }
        q.ro = ld3(C.o) + lens;
        d3 focus_point = ld3(C.o) + dir_base * C.focus_dist;
        q.rd = vnorm(focus_point - q.ro);
        q.time = C.shutter_open + (C.shutter_close - C.shutter_open) * rng.uni();
        q.acc = mk(0.0, 0.0, 0.0);
        q.beta = mk(1.0, 1.0, 1.0);
        q.last_bsdf_pdf = 0.0;
        q.last_non_delta = false;
        q.bounce = 0;
        q.alive = P.max_bounces > 0;
      }
      // the extension ray of every lane, then the shadow rays of the vertices met
      while (q.alive || q.env || q.light) {
        const bool any = q.env || q.light;
        const int which = q.env ? 0 : 1;
        d3 o = q.ro, d = q.rd;
        double tmax = 1e30;
        if (any) {
          o = q.shadow3(which, 0);
          d = q.shadow3(which, 3);
          tmax = q.sh[(which * 10 + 9) * TPT_PLAIN_BLOCK];
        }
        Hit64 hit;
        const bool found = world_hit<G>(P, o, d, q.time, TPT_RAY_EPSILON, tmax, any, st, &hit);
        if (any) {
          if (!found) q.acc = q.acc + q.shadow3(which, 6);
          if (which == 0) q.env = false;
          else q.light = false;
        } else {
          cnt.ext++;
          vertex64(P, q, found, hit, rng, &cnt);
        }
        if (P.shape.mixed || !(q.env || q.light)) break;
      }
      if (!(q.alive || q.env || q.light)) {  // the sample is complete
        const d3 L = q.acc;
        paths++;
        s++;
        // the sums stay in memory (they start at zero): a sample's end is rare, registers are not
        if (writes) {
          double* c = P.acc + 3 * pix;
          c[0] += L.x; c[1] += L.y; c[2] += L.z;
          if (P.acc_sq) {
            double* sq = P.acc_sq + 3 * pix;
            sq[0] += L.x * L.x; sq[1] += L.y * L.y; sq[2] += L.z * L.z;
          }
        }
        n += 1;
        if (P.adaptive) {
          double lum = luminance(L);
          double delta = lum - mean;
          mean += delta / (double)n;
          double delta2 = lum - mean;
          m2 += delta * delta2;
          if (n >= min_spp) {
            double var = n > 1 ? m2 / (double)(n - 1) : __longlong_as_double(0x7ff0000000000000ll);
            double rel = sqrt(var) / fmax(fabs(mean), 1e-4);
            if (rel < P.threshold) done = true;
          }
        }
      }
    }
    if (writes) {
      P.rng[pix] = rng.p.state;
      P.nsamp[pix] = n;
      P.welford[2 * pix] = mean;
      P.welford[2 * pix + 1] = m2;
      P.acc_w[pix] = (double)n;
      if (done) P.done[pix] = 1;
    } else {
      cnt = Count64{0, 0};
      paths = 0;
    }
  }
  // one atomic per wave per counter
  unsigned long long e = cnt.ext, sh = cnt.shadow, pa = paths;
  for (int off = 32; off > 0; off >>= 1) {
    e += (unsigned long long)__shfl_down((long long)e, off);
    sh += (unsigned long long)__shfl_down((long long)sh, off);
    pa += (unsigned long long)__shfl_down((long long)pa, off);
  }
  if (__lane_id() == 0) {
    if (e) atomicAdd((unsigned long long*)&P.stats[0], e);
    if (sh) atomicAdd((unsigned long long*)&P.stats[1], sh);
    if (pa) atomicAdd((unsigned long long*)&P.stats[2], pa);
  }
}

hipError_t launch_plain64(const Plain64Params& P, hipStream_t s) {
  if (P.n_pix <= 0) return hipSuccess;
  const int64_t threads = (int64_t)P.n_pix * (P.shape.quads ? 4 : 1);
  const dim3 grid((uint32_t)((threads + P.shape.lanes - 1) / P.shape.lanes)), block(TPT_PLAIN_BLOCK);
  if (P.shape.quads) hipLaunchKernelGGL(k_plain64<4>, grid, block, 0, s, P);
  else hipLaunchKernelGGL(k_plain64<1>, grid, block, 0, s, P);
  return hipGetLastError();
}

}  // namespace tpt
