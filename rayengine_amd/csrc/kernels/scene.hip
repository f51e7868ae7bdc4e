// Placing the objects' trees in a scene: the flat records as the builder left
// them are copied to the device unchanged, and this kernel rewrites them there
// for their object's place in the scene's arrays.
#include "../internal.hpp"

namespace re {
namespace {

constexpr int kPlaceBlock = 256;
static_assert(sizeof(LeafRec) == sizeof(DevLeaf) && alignof(LeafRec) == alignof(DevLeaf),
              "a leaf record is rewritten in place");

// The blocks of object k follow those of the objects before it (first_block,
// found by bisection, the same in every thread).  Thread i of an object takes
// its node entry, leaf record and triangle record i: entry and leaf references
// and triangle indices are raised by the object's first entry, leaf and
// triangle in the scene (RayEngine/src/World/RTScene.cpp:263-279), prim ids by
// its prim offset, and a leaf record is put in the device's field order, in
// place (both are 64 bytes).  A streaming pass over the records, bound by
// memory; the first object's entries and (without a prim offset) triangles are
// already in place and are not touched.  On the host, record by record into
// concatenated copies, the same made an upload of 521,154 triangle records
// take 12.5 ms; it takes 1.1 ms now, most of it the copies.
__global__ void __launch_bounds__(kPlaceBlock) scene_place_kernel(NodeEntry* __restrict__ nodes,
                                                                  DevLeaf* __restrict__ leaves,
                                                                  TriRec* __restrict__ tris,
                                                                  const ScenePlace* __restrict__ place, int32_t n_obj) {
  int32_t k = 0;
  for (int32_t end = n_obj; end - k > 1;) {
    const int32_t mid = k + (end - k) / 2;
    if (place[mid].first_block <= (int64_t)blockIdx.x) k = mid;
    else end = mid;
  }
  const ScenePlace P = place[k];
  const int64_t i = ((int64_t)blockIdx.x - P.first_block) * kPlaceBlock + threadIdx.x;
  nodes += P.node_base;
  leaves += P.leaf_base;
  tris += P.tri_base;
  if (i < P.n_nodes && (P.node_base | P.leaf_base) != 0) {
    uint32_t meta = nodes[i].meta;
    meta = (meta >> 30) == 3u ? kLeafMeta | ((meta & 0x3fffffffu) + P.leaf_base)
                              : (meta & 0xc0000000u) | ((meta & 0x3fffffffu) + P.node_base);
    nodes[i].meta = meta;
  }
  if (i < P.n_leaves) {
    LeafRec l;
    __builtin_memcpy(&l, leaves + i, sizeof(l));  // not a DevLeaf yet
    for (int f = 0; f < 6; ++f) {
      const int32_t r = l.rope[f];
      if (r != kNoRope) l.rope[f] = ref_is_leaf(r) ? leaf_ref(ref_leaf_id(r) + P.leaf_base) : r + (int32_t)P.node_base;
    }
    l.first += P.tri_base;
    DevLeaf d = dev_leaf(l);
    d.pad[0] = (uint32_t)k;
    leaves[i] = d;
  }
  if (i < P.n_tris && P.prim_offset != 0) tris[i].prim += P.prim_offset;
}

// Leaf records back in the flat field order, for an export.
__global__ void __launch_bounds__(kPlaceBlock) flat_leaves_kernel(const DevLeaf* __restrict__ leaves,
                                                                  LeafRec* __restrict__ out, int64_t n) {
  const int64_t i = (int64_t)blockIdx.x * kPlaceBlock + threadIdx.x;
  if (i < n) out[i] = flat_leaf(leaves[i]);
}

}  // namespace

int64_t scene_place_blocks(const ScenePlace& p) {
  int64_t n = p.n_leaves;
  if ((p.node_base | p.leaf_base) != 0 && p.n_nodes > n) n = p.n_nodes;
  if (p.prim_offset != 0 && p.n_tris > n) n = p.n_tris;
  return (n + kPlaceBlock - 1) / kPlaceBlock;
}

hipError_t launch_scene_place(const DevScene& s, const ScenePlace* place, int32_t n_obj, int64_t blocks,
                              hipStream_t st) {
  if (blocks <= 0) return hipSuccess;
  hipLaunchKernelGGL(scene_place_kernel, dim3((unsigned)blocks), dim3(kPlaceBlock), 0, st, s.nodes, s.leaves, s.tris,
                     place, n_obj);
  return hipGetLastError();
}

hipError_t launch_flat_leaves(const DevLeaf* leaves, LeafRec* out, int64_t n, hipStream_t st) {
  if (n <= 0) return hipSuccess;
  hipLaunchKernelGGL(flat_leaves_kernel, dim3((unsigned)((n + kPlaceBlock - 1) / kPlaceBlock)), dim3(kPlaceBlock), 0,
                     st, leaves, out, n);
  return hipGetLastError();
}

}  // namespace re
