// cn_bvh.h — the 4-wide BVH over world-space triangles that stands in for
// the reference's driver-built TLAS/BLAS pair (gpu/accel.rs:82-163).
#pragma once

#include <stdint.h>

#include <string>
#include <vector>

#include "cn_bvh_split.h"
#include "cn_math.h"
#include "cn_records.h"

namespace cn {

struct WorldTriangle {
    v3 v0, v1, v2;
    uint32_t instance, primitive, flags;
};

struct Bvh4 {
    std::vector<BvhNode4> nodes;  // node 0 is the root and always internal
    std::vector<BvhTriangle> tris;  // leaf order
    uint32_t max_depth = 0;
    double build_seconds = 0.0;
    // The 8-wide collapse of the same binary tree over the same leaves,
    // already quantized (empty when it would be past the limits).
    std::vector<BvhNode8Q> nodes8;
    uint32_t max_depth8 = 0;
};

// A node of the binary tree both builders grow (40 bytes, the layout the
// device builder writes).
struct BinaryNode {
    Box3 box;
    uint32_t left = 0, right = 0;   // children (internal)
    uint32_t first = 0, count = 0;  // leaf range in the builder's order (count > 0)
};
static_assert(sizeof(BinaryNode) == 40, "device and host share this layout");

// What a tree has to keep to: a 4-wide walk's stack takes three entries a
// level and an 8-wide one's seven, and the walks address a node by a 32-bit
// byte offset from the tree's base. LEAF_FIRST_MASK allows 2^27 triangles. By
// BVH_RULES a triangle may be a leaf of its own, and the nodes may number two
// thirds of them; by BVH_COARSE_RULES two triangles never part, a subtree of
// two leaves holds at least three, and the nodes number at most 4/9 of them:
// always fewer than nodes4.
struct BvhLimits {
    uint32_t max_stack;
    uint32_t nodes4 = 1u << 26;
    uint32_t nodes8 = 1u << 25;
};
static_assert(uint64_t(BvhLimits{}.nodes4) * sizeof(BvhNode4Q) <= uint64_t(1) << 32 &&
                  uint64_t(BvhLimits{}.nodes8) * sizeof(BvhNode8Q) <= uint64_t(1) << 32,
              "the last node starts below 2^32");

// Binned-SAH binary build (32 bins on the three axes, leaves by BVH_RULES),
// collapsed to 4-wide nodes by repeatedly opening the child of largest surface
// area. A tree past the limits is grown again by BVH_COARSE_RULES; returns
// false with a message when that is past them too.
bool build_bvh4(const std::vector<WorldTriangle>& input, const BvhLimits& limits, Bvh4* out, std::string* error);

// The collapse step alone, from a binary tree rooted at node 0 (nodes may
// be numbered in any order); max_abs is the scene's largest |coordinate|.
bool collapse_to_bvh4(const std::vector<BinaryNode>& bnodes, float max_abs, const BvhLimits& limits, Bvh4* out,
                      std::string* error);

// The 8-wide collapse of the same binary tree, by the same greedy rule up
// to eight children, straight to BvhNode8Q; fills out->nodes8 and
// max_depth8, or leaves nodes8 empty (returning false) when the tree is past
// the limits.
bool collapse_to_bvh8(const std::vector<BinaryNode>& bnodes, float max_abs, const BvhLimits& limits, Bvh4* out);

// The device-resident outputs of the device builder: device allocations
// the caller takes over (and frees with hipFree); nodes8 is null when the
// 8-wide tree would be past the limits.
struct DeviceBvh {
    BvhTriangle* tris = nullptr;
    BvhNode4Q* nodes = nullptr;
    BvhNode8Q* nodes8 = nullptr;
    uint32_t node_count = 0, node8_count = 0;
};

// A scene's triangles as the device builder reads them: instance i's are the
// mesh triangles from its record's triangle_base on, numbered
// first[i] .. first[i + 1] - 1 in the scene.
struct DeviceTriangles {
    const MeshTriangle* mesh_tris;    // device
    const InstanceRecord* instances;  // device
    const uint32_t* flags;            // host, one word per instance
    const size_t* first;              // host, instance_count + 1
    uint32_t instance_count;
};

// The same trees built entirely on the device (cn_build.hip): top levels by
// device-wide binning with every split decided on the device, subtrees of
// <= 2048 triangles by one workgroup each and of <= 64 by one wave each, the
// collapse to 4- and 8-wide nodes and their quantization on the device, where
// the trees stay (`*dev`); `out` receives the depths and the build time, and
// with `full_nodes` the full-precision 4-wide nodes, which no walk reads.
// Building the same triangles again gives the same records.
bool build_bvh_device(const DeviceTriangles& input, const BvhLimits& limits, bool full_nodes, Bvh4* out,
                      DeviceBvh* dev, std::string* error);

// Rewrites, on the device, the flags word (v2.w) of every leaf-order
// triangle from its instance's entry in `instance_flags` (host array of
// `instances` words): a material edit changes no bounds, so the tree stays.
bool patch_triangle_flags(BvhTriangle* tris, uint32_t count, const uint32_t* instance_flags, uint32_t instances,
                          std::string* error);

// Gathers the pooled mesh triangles hit reconstruction reads, on the device,
// from pooled vertices (host memory, packed xyz positions and normals) and
// pool-wide vertex indices into `triangles` device records.
hipError_t build_mesh_triangles(const float* positions, const float* normals, size_t vertices,
                                const uint32_t* indices, size_t triangles, MeshTriangle* out);

// The packet walk's 128-byte nodes (BvhNode4P) from the device's quantized
// ones, node for node, on the device (the same boxes, planes decoded).
bool decode_packet_nodes(const BvhNode4Q* nodes, uint32_t count, BvhNode4P* out, std::string* error);

// The traversal's 64-byte nodes (BvhNode4Q) from the full-precision ones,
// node for node: each node's grid starts at the low corner of its
// children's union and steps by the smallest power of two that spans the
// union in 255 steps; planes round outward.
void quantize_bvh4(const BvhNode4* nodes, size_t count, BvhNode4Q* out);

}  // namespace cn
