/*
 * vgi_traverse.h — device-side BVH traversal (closest hit and any hit).
 *
 * One lane per ray over the 4-wide BVH of 64-byte quantised nodes.  The
 * traversal stack lives in LDS, interleaved across the 64 lanes of the wave
 * (entry k of lane l at [k*64 + l]) so that a push or pop by all lanes
 * touches 64 consecutive dwords (no bank conflicts).  At a node the hit
 * children are sorted by entry distance and all pushed, farthest first; the
 * next link is then popped.  Boxes are tested with the slab
 * method on the node's 8-bit grid: per axis the ray's distance to grid line
 * q is q * (step / d) + (org - o) / d.  One byte permute turns two planes'
 * bytes into binary16 subnormals q * 2^-24 (exact), and one mixed-precision
 * fused multiply-add per plane (v_fma_mix_f32, a binary16 operand widened
 * exactly) multiplies them by the node's stored step * 2^24.
 *
 * Issue costs that shaped the node step, measured at 8 waves per SIMD in
 * clocks per wave instruction: v_fma_f32, v_mul, v_add, v_mov, v_xor and
 * v_add_u32 2.2-2.4; v_fma_mix, v_perm, conversions, min / max (also the
 * three-operand, integer and f64 ones), compares, conditional moves and
 * three-operand integer instructions 4.1-4.4; anything with a scalar operand
 * at least 4.1.
 */
#pragma once
#include "vgi_bvh.h"

namespace vgi {

// Explicit address spaces for the traversal's memory traffic: the scene
// arrays are global memory and the stack is LDS, also when the scene arrives
// through a pointer loaded from memory (the fused multi-view kernels read it
// from a job table, where the compiler cannot infer the address space and
// would otherwise emit flat accesses that also count against lgkmcnt).
typedef __attribute__((address_space(3))) int32_t* LdsStack;
__device__ __forceinline__ uint32_t lds_addr(LdsStack p) { return (uint32_t)(uintptr_t)p; }
__device__ __forceinline__ __attribute__((address_space(3))) int32_t& lds_at(uint32_t a) { return *(LdsStack)(uintptr_t)a; }
typedef float Vf4 __attribute__((ext_vector_type(4)));
// 16-byte load of scene data (element k of a float4 array) from global memory.
__device__ __forceinline__ Vf4 ld_global16(const void* p, int k) {
    return ((const __attribute__((address_space(1))) Vf4*)p)[k];
}

// The node and triangle arrays are read through buffer descriptors (wave-
// uniform base and size in scalar registers, a 32-bit byte offset per
// lane): the addresses of a node's seven 16-byte loads then cost one 32-bit
// add each instead of 64-bit address arithmetic, and fewer registers.
// Descriptor word 3 of the gfx9 family for untyped dword access; loads
// beyond `bytes` return zeros.  vgi_scene_create keeps both arrays below
// 2^31 bytes.
typedef __amdgpu_buffer_rsrc_t BufRsrc;
__device__ __forceinline__ BufRsrc scene_rsrc(const void* p, uint32_t bytes) {
    return __builtin_amdgcn_make_buffer_rsrc(const_cast<void*>(p), (short)0, (int)bytes, 0x00020000);
}
__device__ __forceinline__ Vf4 ld_buf16(BufRsrc r, uint32_t byte_off) {
    return __builtin_bit_cast(Vf4, __builtin_amdgcn_raw_buffer_load_b128(r, byte_off, 0, 0));
}

struct RayInv {
    f3 o, d, idir;
};

// A direction component of magnitude below 1e-20 gives a finite inverse of
// +-1e20 (slab_nf evaluates P * idir - o * idir, where an infinite inverse
// would turn every plane of that axis into inf - inf = NaN and stop the
// axis from culling anything).  The slab interval of such an axis is then
// (-huge, +huge) for an origin between the planes and empty otherwise, as
// for an exact zero.
__device__ __forceinline__ float safe_dir(float v) { return fabsf(v) < 1e-20f ? copysignf(1e-20f, v) : v; }

__device__ __forceinline__ RayInv make_ray(f3 o, f3 d) {
    RayInv r;
    r.o = o;
    r.d = d;
    r.idir = mk3(1.0f / safe_dir(d.x), 1.0f / safe_dir(d.y), 1.0f / safe_dir(d.z));
    return r;
}

// Byte permute selectors of one axis: they pick the near planes of children
// 0-1 (n01) and 2-3 (n23) from the (hi, lo) word pair, or with the words
// swapped the far ones: near = lo where the direction component is >= 0,
// else hi.  Each byte q gets a zero byte above it and so becomes the
// binary16 subnormal q * 2^-24, exactly.  Choosing the word in the permute
// that widens the bytes costs nothing per node; selecting words first cost
// six conditional moves.  Kernels keep the default binary16 denormal mode
// (inputs and outputs not flushed), which the mixed FMA below relies on.
struct AxisSel {
    uint32_t n01, n23;
};
__device__ __forceinline__ AxisSel axis_sel(bool positive) {
    AxisSel s;
    s.n01 = positive ? 0x0C010C00u : 0x0C050C04u;
    s.n23 = s.n01 ^ 0x00020002u;
    return s;
}
__device__ __forceinline__ uint32_t plane_pair(uint32_t second, uint32_t first, uint32_t sel) {
    return __builtin_amdgcn_perm(second, first, sel);  // selector bytes 0-3: first, 4-7: second
}
// Child k's grid line from the pairs of children 0-1 (p01) and 2-3 (p23),
// as the binary16 q * 2^-24 widened to float (folded into v_fma_mix_f32).
template <int k>
__device__ __forceinline__ float qline(uint32_t p01, uint32_t p23) {
    const uint32_t p = k < 2 ? p01 : p23;
    return (float)__builtin_bit_cast(_Float16, (uint16_t)((k & 1) ? p >> 16 : p & 0xFFFFu));
}

// A ray's near and far plane pairs of one node (children 0-1 and 2-3 per
// axis and side).
struct NodePlanes {
    uint32_t nx01, nx23, fx01, fx23, ny01, ny23, fy01, fy23, nz01, nz23, fz01, fz23;
};

// Slab interval [tn, tf] of child k of a quantised node, clipped to [tmin,
// tmax]; the child is missed unless tn <= tf.  Per axis the distance to grid
// line q is (q * 2^-24) * a + b with a = (step * 2^24) * idir and b =
// (org - o) * idir.  In world units, with u = 2^-24, extent = 255 step and
// plane = org + q * step, the distance errs by at most u * extent (rounding
// of a) + 2 u |org - o| (of the difference and its product) + u |plane - o|
// (of the sum), in all 2 u extent + 3 u (|org| + |o|), besides the relative
// error of idir that all planes of the axis share.  Beyond the padded boxes
// the node's grid boxes hold 8 u max(extent, |org|), more than the node's part
// of that, and 16 u times the scene's reach or half a step (quantise).  So the
// rest, up to 3 u |o|, is covered for origins within five times the reach at
// nodes of a 2000th of it and more, and by the padding (at least 256 u) for
// those within 85 units.  An unused child (lo = 255, hi = 0) has its near plane
// beyond its far one on every axis.
template <int k>
__device__ __forceinline__ void slab_q(f3 a, f3 b, const NodePlanes& p, float tmin, float tmax, float& tn, float& tf) {
    const float tnx = __builtin_fmaf(qline<k>(p.nx01, p.nx23), a.x, b.x);
    const float tfx = __builtin_fmaf(qline<k>(p.fx01, p.fx23), a.x, b.x);
    const float tny = __builtin_fmaf(qline<k>(p.ny01, p.ny23), a.y, b.y);
    const float tfy = __builtin_fmaf(qline<k>(p.fy01, p.fy23), a.y, b.y);
    const float tnz = __builtin_fmaf(qline<k>(p.nz01, p.nz23), a.z, b.z);
    const float tfz = __builtin_fmaf(qline<k>(p.fz01, p.fz23), a.z, b.z);
    tn = fmaxf(fmaxf(fmaxf(tnx, tny), tnz), tmin);
    tf = fminf(fminf(fminf(tfx, tfy), tfz), tmax);
}

__device__ __forceinline__ void count_traversal(const SceneView& s, bool any_hit, uint32_t nodes, uint32_t tris) {
    unsigned long long* c = s.counters + 4u * ((blockIdx.x + 7u * blockIdx.y) % (unsigned)kTraceCounterSlots);
    atomicAdd(c + (any_hit ? 1 : 0), 1ull);
    atomicAdd(c + 2, (unsigned long long)nodes);
    atomicAdd(c + 3, (unsigned long long)tris);
}

// Sort key of a child: its entry distance as the high word of a double and
// its link as the low one, so that one v_min_f64 / v_max_f64 moves both (the
// order of doubles is that of their high words' floats; a finite or infinite
// float there never makes a NaN or signalling pattern).  An exchange is two
// instructions instead of a compare and four conditional moves.
__device__ __forceinline__ double child_key(float t, int32_t link) {
    return __builtin_bit_cast(double, (uint64_t)(uint32_t)link | ((uint64_t)__float_as_uint(t) << 32));
}
__device__ __forceinline__ int32_t key_link(double k) { return (int32_t)__builtin_bit_cast(uint64_t, k); }
// Farther key first.  The instructions themselves: fmin / fmax would first
// canonicalise both operands.
__device__ __forceinline__ void far_first(double& a, double& b) {
    double hi, lo;
    asm("v_max_f64 %0, %1, %2" : "=v"(hi) : "v"(a), "v"(b));
    asm("v_min_f64 %0, %1, %2" : "=v"(lo) : "v"(a), "v"(b));
    a = hi;
    b = lo;
}

// Traversal finished.  Never a leaf link: leaf links are ~(first << 4 | count)
// with first + count <= number of triangles < 2^27.
constexpr int32_t kTraversalDone = INT32_MIN;
__device__ __forceinline__ bool is_leaf(int32_t link) { return (uint32_t)link > (uint32_t)kTraversalDone; }

// One triangle against the ray, without branches (some lane of the wave
// passes almost every test, so an early exit saves nothing): Moller-Trumbore,
// two-sided, in a fixed order of IEEE operations (the oracle's, bit for bit); a
// zero determinant makes u infinite or NaN and fails the conditions.  Updates the hit if
// this one is nearer (ties: the lower triangle id) and says whether it did.
__device__ __forceinline__ bool closer_hit(f3 o, f3 d, Vf4 v0, Vf4 e1v, Vf4 e2v, float tmin, Hit& h) {
    const f3 e1 = mk3(e1v.x, e1v.y, e1v.z), e2 = mk3(e2v.x, e2v.y, e2v.z);
    const f3 pvec = cross3(d, e2);
    const float inv_det = 1.0f / dot3(e1, pvec);
    const f3 tvec = o - mk3(v0.x, v0.y, v0.z);
    const float u = dot3(tvec, pvec) * inv_det;
    const f3 qvec = cross3(tvec, e1);
    const float v = dot3(d, qvec) * inv_det;
    const float t = dot3(e2, qvec) * inv_det;
    const uint32_t id = __float_as_uint(v0.w);
    const bool in = (u >= 0.0f) & (u <= 1.0f) & (v >= 0.0f) & (u + v <= 1.0f) & (t >= tmin);
    const bool hit = in & ((t < h.t) | ((t == h.t) & (id < h.tri)));
    h.t = hit ? t : h.t;
    h.u = hit ? u : h.u;
    h.v = hit ? v : h.v;
    h.tri = hit ? id : h.tri;
    return hit;
}

// Closest hit over [tmin, tmax]; ties in t resolve to the lowest triangle id.
// `stack` points at this lane's slot 0 (stride 64 between entries).
// kCount: the instrumented build (traversal statistics) that adds this ray's
// node and triangle counts to s.counters.
//
// What bounds it: vector instruction issue (while the chip is full), then the
// round trip of each node.  So the wave steps through nodes without a branch
// per child: a step tests four boxes, sorts them, writes all four links to the
// stack (far to near, missed children last, above the new top) and pops its
// next two entries in one LDS read; the second one serves if the first is a
// leaf that is set aside.  A sentinel under the stack ends the ray without a
// test for an empty stack.
//
// A lane sets aside the first leaf it reaches and goes on down the tree.
// The wave takes a node step as long as at least two lanes want one (at a
// node, without a leaf in hand) for every three that hold a leaf; else all
// lanes that hold a leaf intersect it.  Waiting until every lane held one
// ran 30% more node steps on bounce rays, most of them with few lanes, for 20%
// fewer triangle steps; ratios from 1:2 to 3:2 are within 2% of this one.  The
// hits do not depend on the visiting order (closest t, then lowest id), only
// the work does.
//
// A lane whose LDS part is empty takes back what it moved to private memory
// after the wave's next leaf step.  Leaving that until no lane of the wave had
// anything else to do made deep rays finish alone: 256 rays from inside a pile
// of 200,000 quads 447 -> 207 us, a million 2627 -> 2255 us.  It had also kept
// in step waves whose halves cross the pile in opposite directions: those 298
// -> 367 us.  A look at every node step instead costs small frames 0.4%.
// Any-hit rays end early and gain nothing by it (33 -> 31 us); they wait.
//
// Against a step with branches per child and the wait for a leaf in every
// lane: 1M bounce rays on 1M triangles 324 -> 241 us (226 with the present
// tree); the 1080p sampling and spatial passes 1210 -> 995 us; a 1080p frame
// 1951 -> 1687 us, a 256x256 one 617 -> 493 us.  6 or 7 resident waves per SIMD
// instead of 8: within 3%.
template <bool kAnyHit, bool kCount = false>
__device__ __forceinline__ Hit traverse(const SceneView& s, f3 o, f3 d, float tmin, float tmax, LdsStack stack) {
    const RayInv r = make_ray(o, d);
    const AxisSel sx = axis_sel(r.idir.x >= 0.0f), sy = axis_sel(r.idir.y >= 0.0f), sz = axis_sel(r.idir.z >= 0.0f);
    const BufRsrc nodes = scene_rsrc(s.nodes, s.num_nodes * (uint32_t)sizeof(BvhNode));
    const BufRsrc tris = scene_rsrc(s.tris, s.num_tris * (uint32_t)sizeof(BvhTri));
    Hit h;
    h.t = tmax;
    h.u = h.v = 0.0f;
    h.tri = 0xFFFFFFFFu;
    int32_t node = s.root;  // next interior node, a leaf link (while a leaf is held), or kTraversalDone
    int32_t leaf = 0;       // leaf set aside (< 0), 0 for none
    uint32_t n_nodes = 0, n_tris = 0;
    // The stack, by LDS byte address: its top entry is at p + 256, the one
    // below at p.  Slots 0 and 1 are sentinels.
    const uint32_t base = lds_addr(stack);
    uint32_t p = base;
    lds_at(p) = kTraversalDone;
    lds_at(p + 256u) = kTraversalDone;
    // A step writes up to p + 1280.  Where that would leave the LDS part
    // (stack_over) the lane's oldest entries move to private memory.
    static_assert(kStackStride == 256u, "the offsets below");
    int32_t spill[kStackMaxEntries];
    int32_t spilled = 0;
    auto take_back = [&]() {
        if (spilled > 0 && node == kTraversalDone && leaf == 0) {
            spilled -= kSpillEntries;
            for (int k = 0; k < kSpillEntries; ++k) lds_at(base + 256u * (2 + k)) = spill[spilled + k];
            p = base + 256u * (kSpillEntries - 1);
            node = lds_at(p + 512u);
            if (is_leaf(node)) {
                leaf = node;
                node = lds_at(p + 256u);
                p -= 256u;
            }
        }
    };
    // Every step of the wave moves at least one lane, and each node and leaf
    // of a tree is reached at most once per lane (a node has at most 4
    // children); the budget only guards against a corrupted BVH turning into
    // an endless loop.
    uint32_t budget = s.num_nodes < (1u << 23) ? 64u * (5u * s.num_nodes + 8u) : 0xFFFFFFFFu;
    uint64_t m_deep = 0;  // lanes that have moved entries to private memory
    for (;;) {
        const bool inner = node >= 0;
        const uint64_t m_inner = __ballot(inner), m_leaf = __ballot(leaf != 0);
        const uint64_t m_want = m_inner & ~m_leaf;
        if (m_want != 0 && 3 * (int)__popcll(m_want) >= 2 * (int)__popcll(m_leaf)) {
            const uint64_t m_full = full_stacks(m_inner, __ballot(stack_over(p, base)));
            m_deep |= m_full;
            if (m_full != 0) {  // rare
                if (inner && stack_over(p, base)) {
                    if (spilled + kSpillEntries <= (int32_t)kStackMaxEntries) {
                        for (int k = 0; k < kSpillEntries; ++k) spill[spilled + k] = lds_at(base + 256u * (2 + k));
                        spilled += kSpillEntries;
                        p -= 256u * kSpillEntries;
                        // the rest of the slots, in use or not: a loop
                        // over those in use would wait for LDS at each
                        constexpr int kRest = kLdsStackEntries - 2 - kSpillEntries;
                        int32_t rest[kRest];
                        for (int k = 0; k < kRest; ++k) rest[k] = lds_at(base + 256u * (2 + kSpillEntries + k));
                        for (int k = 0; k < kRest; ++k) lds_at(base + 256u * (2 + k)) = rest[k];
                    } else {
                        p = base;  // only for a corrupted BVH: kStackMaxEntries covers every built one
                    }
                }
            }
            if (inner) {
                if (kCount) ++n_nodes;
                const uint32_t nb = (uint32_t)node * (uint32_t)sizeof(BvhNode);
                const Vf4 g0 = ld_buf16(nodes, nb);        // org.xyz, step.x * 2^24
                const Vf4 g1 = ld_buf16(nodes, nb + 16u);  // step.yz * 2^24, q lo.x, q hi.x
                const Vf4 g2 = ld_buf16(nodes, nb + 32u);  // q lo.y, hi.y, lo.z, hi.z
                const Vf4 lk = ld_buf16(nodes, nb + 48u);
                // The links are first needed after the box tests, and left alone
                // the compiler sinks their load to that point: a second round
                // trip per node.  Using them here, and letting nothing cross
                // this point, issues all four loads together.  (Without the
                // barrier the load still sank where registers ran short:
                // 10,000 shadow rays 20.3 -> 21.5 us.)
                __builtin_amdgcn_sched_barrier(0);
                asm volatile("" ::"v"(lk));
                const f3 a = mk3(g0.w * r.idir.x, g1.x * r.idir.y, g1.y * r.idir.z);
                const f3 b = mk3((g0.x - r.o.x) * r.idir.x, (g0.y - r.o.y) * r.idir.y, (g0.z - r.o.z) * r.idir.z);
                const uint32_t lx = __float_as_uint(g1.z), hx = __float_as_uint(g1.w);
                const uint32_t ly = __float_as_uint(g2.x), hy = __float_as_uint(g2.y);
                const uint32_t lz = __float_as_uint(g2.z), hz = __float_as_uint(g2.w);
                const NodePlanes pl{plane_pair(hx, lx, sx.n01), plane_pair(hx, lx, sx.n23),
                                    plane_pair(lx, hx, sx.n01), plane_pair(lx, hx, sx.n23),
                                    plane_pair(hy, ly, sy.n01), plane_pair(hy, ly, sy.n23),
                                    plane_pair(ly, hy, sy.n01), plane_pair(ly, hy, sy.n23),
                                    plane_pair(hz, lz, sz.n01), plane_pair(hz, lz, sz.n23),
                                    plane_pair(lz, hz, sz.n01), plane_pair(lz, hz, sz.n23)};
                float tn0, tn1, tn2, tn3, tf0, tf1, tf2, tf3;
                slab_q<0>(a, b, pl, tmin, h.t, tn0, tf0);
                slab_q<1>(a, b, pl, tmin, h.t, tn1, tf1);
                slab_q<2>(a, b, pl, tmin, h.t, tn2, tf2);
                slab_q<3>(a, b, pl, tmin, h.t, tn3, tf3);
                const bool h0 = tn0 <= tf0, h1 = tn1 <= tf1, h2 = tn2 <= tf2, h3 = tn3 <= tf3;
                const int32_t l0 = __float_as_int(lk.x), l1 = __float_as_int(lk.y);
                const int32_t l2 = __float_as_int(lk.z), l3 = __float_as_int(lk.w);
                if (kAnyHit) {
                    // an occlusion test may visit the hit children in any order
                    lds_at(p + 512u) = l0;
                    p += h0 ? 256u : 0u;
                    lds_at(p + 512u) = l1;
                    p += h1 ? 256u : 0u;
                    lds_at(p + 512u) = l2;
                    p += h2 ? 256u : 0u;
                    lds_at(p + 512u) = l3;
                    p += h3 ? 256u : 0u;
                } else {
                    constexpr float kMiss = -__FLT_MAX__;
                    double k0 = child_key(h0 ? tn0 : kMiss, l0), k1 = child_key(h1 ? tn1 : kMiss, l1);
                    double k2 = child_key(h2 ? tn2 : kMiss, l2), k3 = child_key(h3 ? tn3 : kMiss, l3);
                    far_first(k0, k1);
                    far_first(k2, k3);
                    far_first(k0, k2);
                    far_first(k1, k3);
                    far_first(k1, k2);
                    lds_at(p + 512u) = key_link(k0);
                    lds_at(p + 768u) = key_link(k1);
                    lds_at(p + 1024u) = key_link(k2);
                    lds_at(p + 1280u) = key_link(k3);
                    p += 256u * ((uint32_t)h0 + (uint32_t)h1 + (uint32_t)h2 + (uint32_t)h3);
                }
                const int32_t e0 = lds_at(p + 256u), e1 = lds_at(p);
                const bool aside = (leaf == 0) & is_leaf(e0);
                leaf = aside ? e0 : leaf;
                node = aside ? e1 : e0;
                p -= aside ? 512u : 256u;
            }
        } else if (m_leaf != 0) {
            if (leaf != 0) {
                const uint32_t enc = (uint32_t)(~leaf);
                uint32_t tb = (enc >> 4) * (uint32_t)sizeof(BvhTri);
                const uint32_t end = tb + (enc & 15u) * (uint32_t)sizeof(BvhTri);
                bool hit = false;
                for (; tb != end && !(kAnyHit && hit); tb += (uint32_t)sizeof(BvhTri)) {
                    if (kCount) ++n_tris;
                    hit = closer_hit(o, d, ld_buf16(tris, tb), ld_buf16(tris, tb + 16u), ld_buf16(tris, tb + 32u), tmin,
                                     h);
                }
                leaf = 0;
                if (kAnyHit && hit) {
                    node = kTraversalDone;
                    spilled = 0;
                } else if (is_leaf(node)) {
                    leaf = node;
                    node = lds_at(p + 256u);
                    p -= 256u;
                }
            }
            if (!kAnyHit && m_deep != 0) take_back();
        } else {
            if (__ballot(spilled > 0) == 0) break;  // every lane's stack is empty
            take_back();
        }
        budget = __builtin_amdgcn_readfirstlane(budget) - 1u;
        if (budget == 0u) break;
    }
    if (kCount) count_traversal(s, kAnyHit, n_nodes, n_tris);
    return h;
}

template <bool kCount = false>
__device__ __forceinline__ Hit trace_closest(const SceneView& s, f3 o, f3 d, float tmin, float tmax, LdsStack stack) {
    return traverse<false, kCount>(s, o, d, tmin, tmax, stack);
}
// Shadow ray: true if something is hit on [tmin, tmax] (trace_shadow returns !this).
template <bool kCount = false>
__device__ __forceinline__ bool trace_any(const SceneView& s, f3 o, f3 d, float tmin, float tmax, LdsStack stack) {
    return traverse<true, kCount>(s, o, d, tmin, tmax, stack).tri != 0xFFFFFFFFu;
}

// Per-wave LDS traversal stack: kLdsStackEntries entries x 64 lanes in
// dynamic LDS (launch with traversal_lds_bytes() bytes); deeper entries go to
// private memory.  A ray at a 4-wide node of level d holds at most 3(d+1)
// stacked children, so kStackMaxEntries always suffice there.
#define VGI_TRAVERSAL_STACK(name)                        \
    extern __shared__ int32_t name##_mem[];              \
    LdsStack name = (LdsStack)(name##_mem) + (threadIdx.x & 63u)

}  // namespace vgi
