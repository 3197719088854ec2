/*
 * vgi_bvh.h — software ray tracing on gfx950 (CDNA4 has no ray-tracing
 * hardware): device layout of the scene BVH and the traversal routines that
 * replace violet's VK_KHR_acceleration_structure + TraceRay
 * (restir/raytrace.inc.hlsl:31-56,67-82; render_scene.rs:1170-1712).
 *
 * Layout (built on the host by vgi_bvh.cpp, uploaded once per scene):
 *   nodes : 4-wide BVH, one 64-byte node (half an L2 line, four 16-byte
 *           loads) holds its four children's boxes quantised to 8 bits per
 *           plane on a per-node grid, plane = org + q * step per axis
 *           (stored as step * 2^24, the factor that turns the traversal's
 *           binary16 grid lines q * 2^-24 back into q), and four child
 *           links.  A child link >= 0
 *           is an inner node index; < 0 encodes a leaf ~((first << 4) | n).
 *           A child's quantised box contains its padded box and a margin
 *           for the node's rounding (lo rounded down, hi rounded up).  An unused child has lo = 255, hi = 0 on
 *           every axis (an empty interval) and the empty leaf link ~0.
 *   tris  : leaf-ordered triangles as {v0, e1 = v1-v0, e2 = v2-v0} (3 x
 *           float4, 48 bytes); v0.w carries the scene triangle id.
 * Child boxes are padded, by 2^-16 of the child's coordinates (at least of 1)
 * and on the scales of their node and scene (quantise in vgi_bvh.cpp), so that
 * neither the rounding of the slab test (slab_q in vgi_traverse.h) nor that of
 * the intersection routine prunes a triangle that the routine accepts: the
 * closest hit (smallest t, ties to the lowest triangle id) equals a brute-force
 * loop over all triangles.  Both roundings also grow with the distance to the
 * ray's origin, which no stored box bounds: of 1.2 million hits aimed at the
 * edges of geometry of a unit's size near the origin of a scene of 900 units,
 * none is lost from 1000 units away, 99 from 3000 and 567 from 10,000.
 *
 * Hit semantics follow violet: opaque, two-sided, t in [tmin, tmax];
 * shadow rays accept the first hit (RAY_FLAG_ACCEPT_FIRST_HIT_AND_END_SEARCH).
 */
#pragma once
#include <vector>

#include "../../include/vgi.h"
#include "vgi_common.h"

namespace vgi {

struct BvhNode {
    float org[3];    // grid origin (below every used child's padded box)
    float scale[3];  // grid step per axis times 2^24 (255 steps span the node)
    uint32_t q[6];   // planes lo.x, hi.x, lo.y, hi.y, lo.z, hi.z: byte k = child k
    int32_t link[4];
};
static_assert(sizeof(BvhNode) == 64, "BvhNode layout");

struct BvhTri {
    float4_ v0;  // w = triangle id (bits)
    float4_ e1;
    float4_ e2;
};
static_assert(sizeof(BvhTri) == 48, "BvhTri layout");

// Per-triangle shading data, indexed by scene triangle id.
struct TriShade {
    uint32_t i0, i1, i2;  // vertex indices
    uint32_t material;
};

// MaterialParams (scene_bindings.hlsl:24-51): the layout of vgi_material.
struct Material {
    float base_color[4];
    float metallic;
    float roughness;
    uint32_t color_metalrough_texture;  // base colour | metallic-roughness << 16
    uint32_t normal_texture;            // low 16 bits
};
static_assert(sizeof(Material) == sizeof(vgi_material), "Material layout");

// One material texture on the device: RGBA8 texels (one u32 each, R in the
// low byte) of every mip level, level l at texels + level_offset[l].
constexpr uint32_t kMaxTextureLevels = 16;
struct TexDesc {
    uint32_t width, height, levels, srgb;
    uint32_t level_offset[kMaxTextureLevels];
};
static_assert(sizeof(TexDesc) == 80, "TexDesc layout");
// Texel byte -> float: [0, 256) UNORM (c / 255), [256, 512) the sRGB
// transfer function's inverse, both evaluated in double on the host.
constexpr uint32_t kTexelLutEntries = 512;

struct SceneView {
    const BvhNode* nodes;
    const BvhTri* tris;
    const TriShade* shade;
    const float* positions;  // 3 floats per vertex
    const float* normals;    // 3 floats per vertex
    const Material* materials;
    const float* texcoords;  // 2 floats per vertex, or null
    const float* tangents;   // 4 floats per vertex, or null
    const TexDesc* textures; // the scene's textures (material index - 2)
    const uint32_t* texels;
    const float* texel_lut;  // kTexelLutEntries floats
    uint32_t num_nodes;
    uint32_t num_tris;
    int32_t root;           // link of the root (node 0)
    unsigned long long* counters;  // traversal statistics slots (instrumented kernels only)
};

constexpr float kRayTMin = 0.0005f;  // raytrace.inc.hlsl:39,70
constexpr float kRayTMax = 1000.0f;  // raytrace.inc.hlsl:40,71
constexpr int kBvhMaxDepth = 64;     // binary build depth bound (the 4-wide tree is shallower)

// Traversal stack: kLdsStackEntries entries of each lane live in LDS (two of
// them sentinels, four the room a node step writes before it pops), older
// ones in private (scratch) memory, moved kSpillEntries at a time.  5 KiB per
// one-wave workgroup is the most that leaves LDS (160 KiB per CU) for 32
// resident waves; the scratch part is touched only by rays that hold more
// than 14 entries.
constexpr uint32_t kLdsStackEntries = 20;
constexpr int kSpillEntries = 8;
constexpr uint32_t kStackMaxEntries = 3 * kBvhMaxDepth;  // 3 far children per 4-wide level
constexpr uint32_t kStackStride = 64 * sizeof(int32_t);  // LDS bytes from one entry of a lane to the next
// A node step writes up to p + 5 kStackStride, where p is the byte address
// below the lane's top entry: past the LDS part beyond its slot
// kLdsStackEntries - 6.
VGI_HD bool stack_over(uint32_t p, uint32_t base) { return p > base + kStackStride * (kLdsStackEntries - 6u); }
// The lanes of a wave that move entries to private memory before a node step:
// those at a node (`inner`) whose stack is `over`.  A lane that popped its last
// sentinel is over too: it holds p = base - kStackStride, which wraps for a
// base near zero.  Without the mask every step after a wave's first lane was
// done took the branch of a full stack.
VGI_HD uint64_t full_stacks(uint64_t inner, uint64_t over) { return inner & over; }

// Register budget of the per-pixel ray-tracing kernels, as waves per SIMD:
// 6, 7 and 8 are within 3% of each other (64 registers spill a few values
// outside the traversal loop; 8 waves hide a node's round trip best).  The
// cache-ray pass runs too few waves to gain from it and keeps its registers.
constexpr int kTraceWaves = 8;

// The host side of vgi_scene_create: validation, the binned-SAH build, the
// 4-wide collapse and the device arrays, before any upload (so host tools
// can build and check a scene without a GPU).
struct HostScene {
    std::vector<BvhNode> nodes;
    std::vector<BvhTri> tris;
    std::vector<TriShade> shade;
    std::vector<float> positions, normals, texcoords, tangents;
    std::vector<Material> materials;
    std::vector<TexDesc> textures;
    std::vector<uint32_t> texels;
    std::vector<float> texel_lut;
    int32_t root = 0;
    uint32_t levels = 0;  // levels of 4-wide nodes
};
vgi_status build_scene_host(const vgi_scene_desc* desc, HostScene& out);

// Dynamic LDS bytes of a 64-lane traversal stack.
inline size_t traversal_lds_bytes() { return (size_t)kLdsStackEntries * 64u * sizeof(int32_t); }

struct Hit {
    float t;
    float u, v;  // barycentric weights of vertex 1 and vertex 2
    uint32_t tri;  // scene triangle id; 0xFFFFFFFF = miss
};

}  // namespace vgi
