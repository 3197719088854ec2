// Replays the device traversal (vgi_traverse.h) on the CPU over the nodes that
// the scene builder makes, the node's slab test in the device's float
// operations, against a brute-force loop over all triangles.
//
//   traverse_replay <file>   file: u32 vertices, triangles, rays; f32 positions
//                            [v][3]; u32 indices [t][3]; f32 rays [r][8]
// Prints: rays, hits, lost (closest hit differs from the loop's, bit for bit),
// any (any-hit answer differs).
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

struct Ray {
    f3 o, d;
    float id[3], tmin;
    bool pos[3];
};

float safe_dir(float v) { return std::fabs(v) < 1e-20f ? std::copysign(1e-20f, v) : v; }

// The slab test of child k (slab_q): true if hit, with its entry distance.
bool slab(const Ray& r, const BvhNode& n, int k, float tmax, float& tn) {
    const float o[3] = {r.o.x, r.o.y, r.o.z};
    float tns[3], tfs[3];
    for (int a = 0; a < 3; ++a) {
        const float sa = n.scale[a] * r.id[a];
        const float sb = (n.org[a] - o[a]) * r.id[a];
        const uint32_t lo = (n.q[2 * a] >> (8 * k)) & 255u, hi = (n.q[2 * a + 1] >> (8 * k)) & 255u;
        const float ql = std::ldexp((float)lo, -24), qh = std::ldexp((float)hi, -24);
        tns[a] = std::fmaf(r.pos[a] ? ql : qh, sa, sb);
        tfs[a] = std::fmaf(r.pos[a] ? qh : ql, sa, sb);
    }
    tn = std::fmax(std::fmax(std::fmax(tns[0], tns[1]), tns[2]), r.tmin);
    return tn <= std::fmin(std::fmin(std::fmin(tfs[0], tfs[1]), tfs[2]), tmax);
}

// Nearest child first, or, for any hit, in any order.
RayHit traverse(const HostScene& s, const Ray& r, RayHit h, bool any) {
    std::vector<int32_t> stack{s.root};
    while (!stack.empty()) {
        const int32_t l = stack.back();
        stack.pop_back();
        if (l < 0) {
            const uint32_t enc = ~(uint32_t)l, first = enc >> 4, n = enc & 15u;
            for (uint32_t k = 0; k < n; ++k)
                if (closer_hit(r.o, r.d, s.tris[first + k], r.tmin, h) && any) return h;
            continue;
        }
        const BvhNode& n = s.nodes[l];
        float tn[4];
        int order[4], cnt = 0;
        for (int k = 0; k < 4; ++k)
            if (slab(r, n, k, h.t, tn[k])) order[cnt++] = k;
        std::sort(order, order + cnt, [&](int i, int j) { return tn[i] > tn[j]; });
        for (int i = 0; i < cnt; ++i) stack.push_back(n.link[order[i]]);
    }
    return h;
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

    long long hits = 0, lost = 0, any = 0;
    for (uint32_t k = 0; k < n[2]; ++k) {
        const float* q = rays.data() + 8 * (size_t)k;
        Ray r{mk3(q[0], q[1], q[2]), mk3(q[4], q[5], q[6]), {}, q[3], {}};
        for (int a = 0; a < 3; ++a) {
            r.id[a] = 1.0f / safe_dir(q[4 + a]);
            r.pos[a] = r.id[a] >= 0.0f;
        }
        const RayHit miss{q[7], 0.0f, 0.0f, 0xFFFFFFFFu};
        RayHit brute = miss;
        for (const BvhTri& t : s.tris) closer_hit(r.o, r.d, t, r.tmin, brute);
        const RayHit h = traverse(s, r, miss, false);
        hits += brute.tri != miss.tri;
        lost += std::memcmp(&h, &brute, sizeof(RayHit)) != 0;
        any += (brute.tri != miss.tri) != (traverse(s, r, miss, true).tri != miss.tri);
    }
    std::printf("rays %u hits %lld lost %lld any %lld\n", n[2], hits, lost, any);
    return 0;
}
