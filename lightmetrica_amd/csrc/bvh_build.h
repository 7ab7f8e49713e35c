// Host-side wide-BVH builder for the GPU traversal kernels.
//
// Replaces the reference's two CPU builders:
//   QBVHScene::Build (src/liblightmetrica/scene.qbvh.cpp:453-591): 12-bin SAH on the
//     longest centroid axis, two binary levels per 4-wide node, <= 64-triangle leaves;
//   BVHScene::Build (src/liblightmetrica/scene.bvh.cpp:202-388): pbrt-style 12-bucket SAH.
// This builder bins all three axes (64 bins by default) with a traversal-cost term,
// then collapses the binary tree greedily (largest surface area first) into 4-wide
// nodes laid out for 128-byte cache lines, with leaves of at most 16 triangles
// stored as contiguous 48-byte vertex records.
#pragma once

#include <cstddef>
#include <cstdint>
#include <string>
#include <vector>

namespace lmgpu {

// One 4-wide node: SoA child boxes (96 B) + child references (16 B) + pad = 128 B.
struct alignas(128) Node4 {
    float lo_x[4], hi_x[4], lo_y[4], hi_y[4], lo_z[4], hi_z[4];
    uint32_t child[4];
    uint32_t pad[4];
};
static_assert(sizeof(Node4) == 128, "Node4 must be one 128-byte line");

// The node as the device keeps it: planes are 8-bit steps from `origin`, four children to a word
// (planes[axis][0] the lower, planes[axis][1] the upper ones).
struct alignas(64) NodeQ {
    float origin[3], step[3];
    uint32_t planes[3][2];
    uint32_t child[4];
};
static_assert(sizeof(NodeQ) == 64, "NodeQ is half a 128-byte line");

// Child reference encoding.
constexpr uint32_t kLeafBit = 0x80000000u;
constexpr uint32_t kEmptyChild = 0xffffffffu;
constexpr uint32_t kMaxLeafCount = 16;          // 4-bit count field
constexpr uint32_t kMaxLeafFirst = 0x07ffffffu;  // 27-bit first-record field
inline uint32_t make_leaf_ref(uint32_t first, uint32_t count) {
    return kLeafBit | ((count - 1u) << 27) | first;
}

// Triangle record in leaf order: v0.w carries the scene-order triangle index.
struct alignas(16) TriRecord {
    float v0[4];
    float v1[4];
    float v2[4];
};
static_assert(sizeof(TriRecord) == 48, "TriRecord is 48 bytes");

// The triangle record as the BVH traversal reads it, two to a 128-byte line: v0.w the scene-order
// triangle index, the rest of the fourth column and box_yz the box of the record's leaf as it
// was built (v1.w, v2.w its x range).
struct alignas(64) LeafTri {
    float v0[4], v1[4], v2[4];
    float box_yz[4];  // lo y, hi y, lo z, hi z
};
static_assert(sizeof(LeafTri) == 64, "LeafTri is half a 128-byte line");

// What a traversal reads.  `exact` are the nodes as they were built and `reach` the largest
// coordinate of the scene's box: for the rays that trace_exact (traverse.hpp) decides.
struct BvhDev {
    const NodeQ* nodes;
    const LeafTri* tris;
    const Node4* exact;
    float reach;
};

// Affine-transform record of a triangle for the path tracer of scenes small enough to test
// every triangle per ray (Baldwin and Weber, "Fast Ray-Triangle Intersections by Coordinate
// Transformation", JCGT 5(3), 2016): rows r0, r1, r2 (xyz linear part, w offset) of the map
// that takes the triangle's vertices v0, v1, v2 to (0,0,0), (1,0,0), (0,1,0) and the axis of
// the normal's largest component to (0,0,1).  A point p of the ray lies on the triangle's plane
// where r2 . p + r2.w = 0, and then (r0 . p + r0.w, r1 . p + r1.w) are the weights of v1 and
// v2.  `id` is the scene-order triangle index.  A degenerate triangle gets r2 = (0, 0, 0, 1),
// which no ray meets.
struct alignas(16) XformRecord {
    float r0[4], r1[4], r2[4];
    uint32_t id, pad[3];
};
static_assert(sizeof(XformRecord) == 64, "XformRecord is 64 bytes");

// The XformRecord of every TriRecord (in the same order), computed in double precision.
std::vector<XformRecord> make_xform_records(const std::vector<TriRecord>& tris);

struct BuildParams {
    uint32_t max_leaf_size = 4;
    uint32_t bins = 64;
    float traversal_cost = 1.2f;
    int num_threads = 0;
    // Binary-tree depth from which nodes split at the object median of the longest centroid
    // axis instead of by SAH (build_wide_bvh lowers it when a tree comes out too deep).
    uint32_t median_depth = 0xffffffffu;
};

// The deepest 4-wide tree the traversal stack holds (three pushes per level in 96 slots).
constexpr uint32_t kMaxWideDepth = 32;
// The most nodes a tree may have: the traversal addresses node words by 32-bit byte offsets.
constexpr uint32_t kMaxNodes = 1u << 25;

struct WideBVH {
    std::vector<Node4> nodes;
    std::vector<TriRecord> tris;
    uint32_t num_leaves = 0;
    uint32_t max_depth = 0;  // inner-node levels on the deepest root-to-leaf path
    uint32_t median_depth = 0xffffffffu;  // the BuildParams::median_depth the tree was built with
    double sah_cost = 0.0;
    double build_seconds = 0.0;
};

// Places the leaves of `bvh` for the device: pad[slot] of a node becomes the first LeafTri of the
// leaf in that child slot.  A leaf of two or more records starts on a line, so that it takes no
// more lines than it fills, unless the padded array would outgrow the 27-bit leaf offsets.
// Returns the number of LeafTri.
uint32_t place_leaves(WideBVH& bvh);

// positions: 3 floats per vertex; faces: 3 indices per triangle.
// Returns false with `err` set when the input cannot be built.  A tree deeper than
// kMaxWideDepth (strongly clustered geometry, where SAH peels one cluster off per level) is
// rebuilt with object-median splits from a shallower binary depth on, down to an all-median
// tree, whose depth is at most log2 of the triangle count.
bool build_wide_bvh(const float* positions, uint32_t num_vertices, const uint32_t* faces, uint32_t num_triangles,
                    const BuildParams& params, WideBVH& out, std::string& err);

}  // namespace lmgpu
