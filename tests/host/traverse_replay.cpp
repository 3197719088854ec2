// Replays the device traversal (vgi_traverse.h) on the CPU over the nodes that
// the scene builder makes: a wave of 64 rays in lockstep with its traversal
// stack in a 20-entry "LDS" part and a private part, the node's slab test in
// the device's float operations, against a brute-force loop over all
// triangles.  Reports the rays whose closest hit differs from the loop's and
// how the stacks grew; an access outside a stack ends the program.
//
//   traverse_replay <file>   file: u32 vertices, triangles, rays; f32 positions
//                            [v][3]; u32 indices [t][3]; f32 rays [r][8]
// Prints: rays, hits, lost (closest hit differs), any (any-hit answer differs),
// the most stack entries of a lane, the most moves to private memory of a lane,
// node steps of all waves, how many of them did stack moves, how many had a
// lane with entries to move, and the node steps with all of every stack in LDS.
#include <algorithm>
#include <cmath>
#include <cstdint>
#include <cstdio>
#include <cstdlib>
#include <cstring>
#include <vector>

#include "vgi_bvh.h"
#include "vgi_internal.h"

using namespace vgi;

namespace {

constexpr int32_t kDone = INT32_MIN;
bool is_leaf(int32_t l) { return (uint32_t)l > (uint32_t)kDone; }

void require(bool ok, const char* what) {
    if (!ok) {
        std::fprintf(stderr, "traverse_replay: %s\n", what);
        std::exit(2);
    }
}

struct RayHit {
    float t, u, v;
    uint32_t tri;
};

bool closer_hit(f3 o, f3 d, const BvhTri& tr, float tmin, RayHit& h) {
    const f3 e1 = mk3(tr.e1.x, tr.e1.y, tr.e1.z), e2 = mk3(tr.e2.x, tr.e2.y, tr.e2.z);
    const f3 pvec = cross3(d, e2);
    const float inv_det = 1.0f / dot3(e1, pvec);
    const f3 tvec = o - mk3(tr.v0.x, tr.v0.y, tr.v0.z);
    const float u = dot3(tvec, pvec) * inv_det;
    const f3 qvec = cross3(tvec, e1);
    const float v = dot3(d, qvec) * inv_det;
    const float t = dot3(e2, qvec) * inv_det;
    uint32_t id;
    std::memcpy(&id, &tr.v0.w, 4);
    const bool in = (u >= 0.0f) && (u <= 1.0f) && (v >= 0.0f) && (u + v <= 1.0f) && (t >= tmin);
    if (!in || !(t < h.t || (t == h.t && id < h.tri))) return false;
    h = RayHit{t, u, v, id};
    return true;
}

struct Totals {
    long long steps = 0, move_steps = 0, needed_steps = 0;
    int max_entries = 0, max_moves = 0;
};

struct Lane {
    bool used = false;
    f3 o, d;
    float id[3], tmin;
    bool pos[3];
    RayHit h;
    int32_t node, leaf = 0;
    uint32_t base, p;
    std::vector<int32_t> lds;
    int32_t spill[kStackMaxEntries];
    int spilled = 0, moves = 0;
    int32_t& at(uint32_t a) {
        const uint32_t off = a - base;
        require(off % kStackStride == 0 && off / kStackStride < lds.size(), "LDS stack access out of range");
        return lds[off / kStackStride];
    }
    int entries() const { return (int32_t)(p - base) / (int32_t)kStackStride + spilled; }
};

float safe_dir(float v) { return std::fabs(v) < 1e-20f ? std::copysign(1e-20f, v) : v; }

// The slab test of child k (slab_q): true if hit, with its entry distance.
bool slab(const Lane& l, const BvhNode& n, int k, float& tn) {
    const float o[3] = {l.o.x, l.o.y, l.o.z};
    float near = l.tmin, far = l.h.t, tns[3], tfs[3];
    for (int a = 0; a < 3; ++a) {
        const float sa = n.scale[a] * l.id[a];
        const float sb = (n.org[a] - o[a]) * l.id[a];
        const uint32_t lo = (n.q[2 * a] >> (8 * k)) & 255u, hi = (n.q[2 * a + 1] >> (8 * k)) & 255u;
        const float ql = std::ldexp((float)lo, -24), qh = std::ldexp((float)hi, -24);
        tns[a] = std::fmaf(l.pos[a] ? ql : qh, sa, sb);
        tfs[a] = std::fmaf(l.pos[a] ? qh : ql, sa, sb);
    }
    near = std::fmax(std::fmax(std::fmax(tns[0], tns[1]), tns[2]), near);
    far = std::fmin(std::fmin(std::fmin(tfs[0], tfs[1]), tfs[2]), far);
    tn = near;
    return near <= far;
}

// Nothing left but entries in private memory.
bool waits(const Lane& l) { return l.used && l.spilled > 0 && l.node == kDone && l.leaf == 0; }

// `bounded`: with the stack in two parts; else all of it in "LDS".
template <bool kAny>
void run_wave(const HostScene& s, std::vector<Lane>& w, Totals& totals, bool bounded = true) {
    for (Lane& l : w) {
        l.lds.assign(bounded ? kLdsStackEntries : kStackMaxEntries + 8, 0);
        l.p = l.base;
        l.at(l.p) = kDone;
        l.at(l.p + kStackStride) = kDone;
        l.node = s.root;
    }
    bool deep = false;
    for (;;) {
        int n_leaf = 0, n_want = 0;
        for (const Lane& l : w) {
            if (!l.used) continue;
            n_leaf += l.leaf != 0;
            n_want += l.node >= 0 && l.leaf == 0;
        }
        if (n_want != 0 && 3 * n_want >= 2 * n_leaf) {
            ++totals.steps;
            uint64_t inner = 0, over = 0;
            bool need = false;
            for (size_t k = 0; k < w.size(); ++k) {
                const Lane& l = w[k];
                if (!l.used) continue;
                inner |= (uint64_t)(l.node >= 0) << k;
                over |= (uint64_t)(bounded && stack_over(l.p, l.base)) << k;
                need |= bounded && l.node >= 0 && (int32_t)(l.p - l.base) > (int32_t)(kStackStride * (kLdsStackEntries - 6));
            }
            totals.move_steps += full_stacks(inner, over) != 0;
            totals.needed_steps += need;
            for (Lane& l : w) {
                if (!l.used || l.node < 0) continue;
                if (bounded && stack_over(l.p, l.base)) {
                    require(l.spilled + kSpillEntries <= (int)kStackMaxEntries, "private stack full");
                    for (int k = 0; k < kSpillEntries; ++k) l.spill[l.spilled + k] = l.at(l.base + kStackStride * (2 + k));
                    l.spilled += kSpillEntries;
                    deep = true;
                    l.p -= kStackStride * kSpillEntries;
                    constexpr int kRest = kLdsStackEntries - 2 - kSpillEntries;
                    for (int k = 0; k < kRest; ++k)
                        l.at(l.base + kStackStride * (2 + k)) = l.at(l.base + kStackStride * (2 + kSpillEntries + k));
                    if (++l.moves > totals.max_moves) totals.max_moves = l.moves;
                }
                const BvhNode& n = s.nodes[l.node];
                float tn[4];
                bool hit[4];
                int order[4] = {0, 1, 2, 3}, cnt = 0;
                for (int k = 0; k < 4; ++k) {
                    hit[k] = slab(l, n, k, tn[k]);
                    cnt += hit[k];
                }
                if (!kAny)  // farther first, missed children last
                    for (int i = 0; i < 3; ++i)
                        for (int j = i + 1; j < 4; ++j) {
                            const float ti = hit[order[i]] ? tn[order[i]] : -INFINITY;
                            const float tj = hit[order[j]] ? tn[order[j]] : -INFINITY;
                            if (tj > ti) std::swap(order[i], order[j]);
                        }
                if (kAny) {
                    for (int k = 0; k < 4; ++k) {
                        l.at(l.p + 2 * kStackStride) = n.link[k];
                        l.p += hit[k] ? kStackStride : 0u;
                    }
                } else {
                    for (int k = 0; k < 4; ++k) l.at(l.p + (2 + k) * kStackStride) = n.link[order[k]];
                    l.p += kStackStride * cnt;
                }
                totals.max_entries = std::max(totals.max_entries, l.entries());
                const int32_t e0 = l.at(l.p + kStackStride), e1 = l.at(l.p);
                const bool aside = l.leaf == 0 && is_leaf(e0);
                l.leaf = aside ? e0 : l.leaf;
                l.node = aside ? e1 : e0;
                l.p -= aside ? 2 * kStackStride : kStackStride;
            }
        } else {
            bool left = n_leaf != 0;
            for (const Lane& l : w) left |= l.used && l.spilled > 0;
            if (!left) break;
            for (Lane& l : w) {
                if (!l.used || l.leaf == 0) continue;
                const uint32_t enc = ~(uint32_t)l.leaf, first = enc >> 4, n = enc & 15u;
                bool got = false;
                for (uint32_t k = 0; k < n && !(kAny && got); ++k)
                    got = closer_hit(l.o, l.d, s.tris[first + k], l.tmin, l.h) || (!kAny && got);
                l.leaf = 0;
                if (kAny && got) {
                    l.node = kDone;
                    l.spilled = 0;
                } else if (is_leaf(l.node)) {
                    l.leaf = l.node;
                    l.node = l.at(l.p + kStackStride);
                    l.p -= kStackStride;
                }
            }
            if (deep && (!kAny || n_leaf == 0))
                for (Lane& l : w)
                    if (waits(l)) {
                        l.spilled -= kSpillEntries;
                        for (int k = 0; k < kSpillEntries; ++k) l.at(l.base + kStackStride * (2 + k)) = l.spill[l.spilled + k];
                        l.p = l.base + kStackStride * (kSpillEntries - 1);
                        l.node = l.at(l.p + 2 * kStackStride);
                        if (is_leaf(l.node)) {
                            l.leaf = l.node;
                            l.node = l.at(l.p + kStackStride);
                            l.p -= kStackStride;
                        }
                    }
        }
    }
    for (const Lane& l : w) require(!l.used || l.spilled == 0, "a lane ended with entries in private memory");
}

template <class T>
std::vector<T> read(std::FILE* f, size_t n) {
    std::vector<T> v(n);
    require(std::fread(v.data(), sizeof(T), n, f) == n, "short input");
    return v;
}

}  // namespace

int main(int argc, char** argv) {
    require(argc == 2, "usage: traverse_replay <file>");
    std::FILE* f = std::fopen(argv[1], "rb");
    require(f != nullptr, "cannot open the input");
    const std::vector<uint32_t> n = read<uint32_t>(f, 3);
    const std::vector<float> pos = read<float>(f, 3 * (size_t)n[0]);
    const std::vector<uint32_t> idx = read<uint32_t>(f, 3 * (size_t)n[1]);
    const std::vector<float> rays = read<float>(f, 8 * (size_t)n[2]);
    std::fclose(f);
    vgi_material mat{};
    vgi_scene_desc desc{};
    desc.positions = pos.data();
    desc.num_vertices = n[0];
    desc.indices = idx.data();
    desc.num_triangles = n[1];
    desc.materials = &mat;
    desc.num_materials = 1;
    HostScene s;
    require(build_scene_host(&desc, s) == VGI_OK, "scene refused");

    Totals totals, unbounded;
    long long hits = 0, lost = 0, any = 0;
    for (uint32_t r0 = 0; r0 < n[2]; r0 += 64) {
        std::vector<Lane> w(64);
        for (uint32_t k = 0; k < 64; ++k) {
            Lane& l = w[k];
            l.base = 4 * k;  // LDS byte address of the lane's slot 0 in a kernel without other LDS
            l.used = r0 + k < n[2];
            if (!l.used) continue;
            const float* r = rays.data() + 8 * (size_t)(r0 + k);
            l.o = mk3(r[0], r[1], r[2]);
            l.d = mk3(r[4], r[5], r[6]);
            l.tmin = r[3];
            l.h = RayHit{r[7], 0.0f, 0.0f, 0xFFFFFFFFu};
            for (int a = 0; a < 3; ++a) {
                l.id[a] = 1.0f / safe_dir(r[4 + a]);
                l.pos[a] = l.id[a] >= 0.0f;
            }
        }
        std::vector<RayHit> brute(64);
        for (int k = 0; k < 64; ++k) {
            brute[k] = w[k].h;
            if (w[k].used)
                for (const BvhTri& t : s.tris) closer_hit(w[k].o, w[k].d, t, w[k].tmin, brute[k]);
        }
        const std::vector<Lane> start = w;
        std::vector<Lane> wa = w, whole = w;
        run_wave<false>(s, w, totals);
        run_wave<true>(s, wa, totals);
        run_wave<false>(s, whole, unbounded, false);
        run_wave<true>(s, whole = start, unbounded, false);
        for (int k = 0; k < 64; ++k) {
            if (!w[k].used) continue;
            const bool hit = brute[k].tri != 0xFFFFFFFFu;
            hits += hit;
            lost += std::memcmp(&w[k].h, &brute[k], sizeof(RayHit)) != 0;
            any += hit != (wa[k].h.tri != 0xFFFFFFFFu);
        }
    }
    std::printf("rays %u hits %lld lost %lld any %lld max_entries %d max_moves %d steps %lld move_steps %lld "
                "needed_steps %lld unbounded_steps %lld nodes %zu\n",
                n[2], hits, lost, any, totals.max_entries, totals.max_moves, totals.steps, totals.move_steps,
                totals.needed_steps, unbounded.steps, s.nodes.size());
    return 0;
}
