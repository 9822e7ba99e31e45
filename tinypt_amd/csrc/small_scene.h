// small_scene.h -- which scenes the small-scene kernels take (host arithmetic).
#pragma once

#include <stdint.h>

namespace tpt {

// A scene whose rays all stay in world space and whose trees fit a corner of the LDS: the traversal
// kernels for it keep nodes, triangles, spheres and items there (SmallTree).
struct SmallScene {
  uint32_t node0, n_nodes, tri0, n_tris, n_items, n_sph;
  int32_t flat_root;  // the flattened tree's root (none: TPT_REF_EMPTY)
  uint32_t stack;     // traversal stack entries a lane can need
  uint32_t bytes;     // LDS bytes of the scene; 0: the scene is not small
};
#define TPT_SMALL_NODE_BYTES 112   // a Node4 without its padding; seven 16 B groups spread its fields over the banks
// Scene data that the small-scene kernels take, measured on both sides (512^2 x 64 spp, 12 bounces,
// these kernels against one ray per lane on device memory): mesh of 82 triangles, 7 KB, 5.19 ->
// 4.53 ms; 322 triangles, 27 KB, 5.97 -> 5.65 ms.  Beyond, the scene and the stacks leave two blocks
// a CU, and the gain, already falling with the longer rays, ends.
#define TPT_SMALL_MAX_BYTES 32768
#define TPT_SMALL_MAX_STACK 20     // entries
inline uint32_t small_scene_bytes(uint32_t nodes, uint32_t tris, uint32_t items, uint32_t sph) {
  return (nodes * TPT_SMALL_NODE_BYTES + tris * 48u + sph * 32u + (tris + items) * 4u + 15u) / 16u * 16u;
}

// Whether SmallTree can address the scene's nodes and triangles: it keeps their places in the scene's own
// arrays, behind those of meshes that no instance uses, and offsets them by 32-bit signed bytes.
inline bool small_scene_addressable(const SmallScene& m) {
  return ((uint64_t)m.node0 + m.n_nodes) * TPT_SMALL_NODE_BYTES <= INT32_MAX &&
         ((uint64_t)m.tri0 + m.n_tris) * 48 <= INT32_MAX;
}

// LDS of a block of `block` threads: the scene and the lanes' stacks.
inline uint32_t small_lds(const SmallScene& m, uint32_t block) { return m.bytes + m.stack * block * 4; }

}  // namespace tpt
