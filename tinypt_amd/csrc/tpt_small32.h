// tpt_small32.h -- small scenes: the FP32 trees in LDS.
#pragma once

#include <hip/hip_runtime.h>
#include <stdint.h>

#include "small_scene.h"
#include "tpt_trace32.h"

namespace tpt {

struct SmallTree {
  static constexpr bool kWorldOnly = true;
  const char *nodes, *tris, *sph;  // LDS, offset so that the scene's own indices address them
  const int32_t *inst, *items;
  int32_t root;
  __device__ __forceinline__ uint32_t node(int32_t ref) const { return (uint32_t)ref * TPT_SMALL_NODE_BYTES; }
  __device__ __forceinline__ float4 planes(uint32_t at) const { return *reinterpret_cast<const float4*>(nodes + (int32_t)at); }
  __device__ __forceinline__ int4 children(uint32_t at) const {
    return *reinterpret_cast<const int4*>(nodes + (int32_t)(at + 96u));
  }
  __device__ __forceinline__ const float4* tri(uint32_t slot) const {
    return reinterpret_cast<const float4*>(tris + (int32_t)(slot * 48u));
  }
  __device__ __forceinline__ int32_t tri_inst(uint32_t slot) const { return inst[(int32_t)slot]; }
  __device__ __forceinline__ int32_t item(uint32_t k) const { return items[k]; }
  __device__ __forceinline__ const double* sphere(int32_t s) const { return reinterpret_cast<const double*>(sph + s * 32); }
  __device__ __forceinline__ int32_t flat_root() const { return root; }
};

// Copies the scene into `mem` (every thread of a block of BLOCK threads must call it) and returns its
// trees and, in *stack, this lane's stack behind them.
template <uint32_t BLOCK>
__device__ __forceinline__ SmallTree load_small(const SceneF32& S, const SmallScene& m, float4* mem, LaneStackT<false>* stack) {
  float4* tris = mem + m.n_nodes * (TPT_SMALL_NODE_BYTES / 16);
  float4* sph = tris + m.n_tris * 3;
  int32_t* inst = reinterpret_cast<int32_t*>(sph + m.n_sph * 2);
  int32_t* items = inst + m.n_tris;
  const float4* gn = reinterpret_cast<const float4*>(S.nodes + m.node0);
  for (uint32_t i = threadIdx.x; i < m.n_nodes * 7; i += BLOCK) mem[i] = gn[i / 7 * 8 + i % 7];
  const float4* gt = reinterpret_cast<const float4*>(S.tris + m.tri0);
  for (uint32_t i = threadIdx.x; i < m.n_tris * 3; i += BLOCK) tris[i] = gt[i];
  const float4* gs = reinterpret_cast<const float4*>(S.sph);
  for (uint32_t i = threadIdx.x; i < m.n_sph * 2; i += BLOCK) sph[i] = gs[i];
  for (uint32_t i = threadIdx.x; i < m.n_tris; i += BLOCK) inst[i] = S.tri_inst[m.tri0 + i];
  for (uint32_t i = threadIdx.x; i < m.n_items; i += BLOCK) items[i] = S.tlas_items[i];
  __syncthreads();
  *stack = LaneStackT<false>{reinterpret_cast<int32_t*>(mem + m.bytes / 16) + threadIdx.x, nullptr, (int)BLOCK,
                             (int)m.stack};
  return SmallTree{reinterpret_cast<const char*>(mem) - m.node0 * TPT_SMALL_NODE_BYTES,
                   reinterpret_cast<const char*>(tris) - m.tri0 * 48u, reinterpret_cast<const char*>(sph),
                   inst - m.tri0, items, m.flat_root};
}

}  // namespace tpt
