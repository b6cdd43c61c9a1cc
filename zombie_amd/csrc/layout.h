// layout.h -- packed scene layout shared by the host builder and the gfx950 kernels.
//
// Wide BVH node (W = 4 or 8 children), structure of arrays inside the node so that one
// lane streams a node with W*2*DIM/4 + W/4 dwordx4 loads:
//   float lo[DIM][W]; float hi[DIM][W]; int32 child[W]; padding to NODE_BYTES.
// child >= 0 : index of an inner node
// child <  0 : leaf, ~child = (first_prim << 4) | (prim_count - 1)
// empty slots hold a degenerate box at +1e30 whose squared distance overflows to +inf and whose slab
// interval lies beyond any ray within the scene, so traversal does not enter them.  It would where a
// comparison says nothing: a NaN coordinate (fmaxf(NaN, 0) is 0), or a ray of unbounded length along a
// diagonal.  Their code is therefore that of a leaf, the first primitive alone, which is harmless to
// test; the code of an inner node would lead back into the tree and the traversal would not end.
//
// Primitives are stored in leaf order:
//   3D triangle : 12 floats  a.xyz b.xyz c.xyz, caller index (int bits), 0, 0   (48 B)
//   2D segment  :  4 floats  a.xy b.xy                                          (16 B)
//                 + int32 caller index in a separate array
#pragma once
#include <hip/hip_runtime.h>

#include <cstdint>

namespace zg {

constexpr float kEmptyBox = 1e30f;
constexpr int kEmptyChild = ~0;   // encodeLeaf(0, 1)

template <int DIM, int W>
struct NodeLayout {
    static constexpr int kBoxFloats = 2 * DIM * W;
    static constexpr int kRawFloats = kBoxFloats + W;
    // pad to a multiple of 64 bytes (16 floats)
    static constexpr int kFloats = ((kRawFloats + 15) / 16) * 16;
    static constexpr int kBytes = kFloats * 4;
    static constexpr int kChildOffset = kBoxFloats;
    static constexpr __host__ __device__ bool emptySlot(const float* node, int k) { return node[k] >= 0.1f * kEmptyBox; }
};

// Oriented boxes of the same tree (same node indices, child slots and child codes), read by exact
// closest-point queries: node n holds its W children one after the other,
//   3D  64 B: centre.xyz, code; axis0.xyz, half0; axis1.xyz, half1; axis2.xyz, half2
//   2D  32 B: centre.xy, axis0.xy; half0, half1 (axis1 = axis0 turned by 90 degrees), code, 0
// An empty slot has half extents of -kEmptyBox: its distance overflows to +inf (its code: kEmptyChild).
template <int DIM>
struct ObbLayout {
    static constexpr int kVec = DIM == 3 ? 4 : 2;   // float4 per child
};

// Entry nodes.  An exact query of a walk knows a primitive close to its point x: the closest one of the query
// before (the seed), at distance s.  Whatever is closest to x lies within s of x, hence within 2 s of the
// seed.  For every leaf, kEntryLevels more nodes of oriented boxes after the BVH's own (indices nNodes +
// leaf * kEntryLevels + level) hold a cover, in at most W items, of everything within reach_level =
// kEntryReach * diagonal of the leaf's box * kEntryRatio^level of that box; the query starts at the smallest
// level with 2 s <= reach_level instead of at the root.  primEntry holds, for every packed primitive,
// (reach_0 / 2)^2 and (int bits) the level-0 entry of its leaf.
//
// Node visits per query on the 81,920-triangle sphere 12.7 -> 8.8, 100,000 points x 64 walks 66.0 -> 58.5 ms;
// 12 screened instances 61.3 -> 58.0 ms, 1,024 segments in 2D 13.5 -> 13.1 ms.  Levels x reach x ratio of
// 4 x 0.25 x 4 / 3 x 0.25 x 4 / 2 x 0.5 x 8 / 4 x 0.1 x 4 ran 57.9 / 57.4 / 58.5 / 57.1 ms there: two
// levels need half of four's memory (W * 64 B a level and leaf in 3D) for 1-2%.
constexpr int kEntryLevels = 2;
constexpr float kEntryReach = 0.5f;
constexpr float kEntryRatio = 8.0f;

template <int DIM>
struct PrimLayout {
    static constexpr int kFloats = DIM == 3 ? 12 : 4;
    static constexpr int kBytes = kFloats * 4;
};

// silhouette candidate (2D reflecting boundary): v.xy, n0.xy, n1.xy, single-neighbour flag, pad
constexpr int kSilFloats = 8;    // 2D candidate: vertex.xy, n0.xy, n1.xy, open end, pad
constexpr int kSil3Floats = 16;  // 3D candidate edge: a.xyz, open edge; b.xyz, 0; n0.xyz, 0; n1.xyz, 0

inline int leafFirst(int child) { return (~child) >> 4; }
inline int leafCount(int child) { return ((~child) & 15) + 1; }
inline int encodeLeaf(int first, int count) { return ~((first << 4) | (count - 1)); }

// Device view of one boundary part (absorbing or reflecting)
struct BoundaryView {
    const float* nodes;    // nNodes * NodeLayout::kFloats
    const float* prims;    // nPrims * PrimLayout::kFloats (leaf order)
    const int32_t* primIds;// 2D: caller index per packed primitive
    const float* sil;      // reflecting: silhouette candidates (kSilFloats each in 2D, kSil3Floats in 3D)
    const float* silNodes; // reflecting: wide BVH over the silhouette candidates
    const float* silCones; // per silhouette-BVH child: normal cone (2D: axis.xy, sin, cos of half-angle + margin;
                           // 3D: axis.xyz, sin; cos, 0, 0, 0)
    float silConePrecision;// the silhouette precision the cones' margin covers
    const float* robinMax; // 2D reflecting: largest Robin coefficient per packed primitive (null: 0)
    const float4* obb;     // absorbing: nNodes * W oriented child boxes, then the entry nodes (null: queries
                           // use the nodes' boxes)
    const float2* primEntry;  // absorbing, with obb: entry record per packed primitive
    int32_t nNodes;
    int32_t nPrims;
    int32_t nSil;
    int32_t nSilNodes;
};

struct SceneView {
    BoundaryView abs, refl;
    float dmin[3], dmax[3];
    int32_t dim, width;
};

}  // namespace zg
