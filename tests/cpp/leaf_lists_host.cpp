// Host build of the mesh queries (rocketsim_amd/csrc/rsg_mesh.h) for
// tests/test_leaf_lists.py: the same query answered by the leaf lists and by
// the tree walk.
#include <cstring>
#include <vector>

#include "../../rocketsim_amd/csrc/rsg_mesh_build.h"

using namespace rsg;

namespace {
// Triangles whose own box touches the query box, in the order reported.
struct BoxHits {
    const MeshView* m;
    V3 lo, hi;
    std::vector<int> t;
    void operator()(int tri) {
        V3 v[3];
        mesh_triangle(*m, tri, v);
        if (triangle_aabb_overlap(v, lo, hi)) t.push_back(tri);
    }
};
// Closest hit of a ray and the triangles that became it, in order.
struct RayHits {
    const MeshView* m;
    V3 from, to;
    float frac;
    V3 n;
    std::vector<int> t;
    void operator()(int tri) {
        V3 v[3];
        mesh_triangle(*m, tri, v);
        if (ray_triangle(from, to, v[0], v[1], v[2], frac, n)) t.push_back(tri);
    }
};
}  // namespace

extern "C" {

void* ll_mesh(const void* cmf, uint64_t size) {
    auto* m = new HostMesh();
    if (!build_host_mesh(cmf, size, *m).empty()) { delete m; return nullptr; }
    return m;
}
void ll_free(void* m) { delete (HostMesh*)m; }
void ll_bounds(void* p, float* out) {
    const HostMesh& m = *(HostMesh*)p;
    std::memcpy(out, &m.aabb_min, 12);
    std::memcpy(out + 3, &m.aabb_max, 12);
}
int ll_has_lists(void* p) {
    const MeshView v = ((HostMesh*)p)->view();
    return (v.box_grid.items ? 1 : 0) + (v.ray_grid.items ? 2 : 0);
}

// Over n boxes (lo, hi): how many the lists served, and -1 if any answer
// differs from the tree's.  *n_hits: triangles reported in all.
int ll_boxes(void* p, int n, const float* boxes, long* n_hits) {
    const MeshView with = ((HostMesh*)p)->view();
    MeshView without = with;
    without.box_grid.items = nullptr;
    int served = 0;
    for (int i = 0; i < n; i++) {
        const V3 lo = v3(boxes[6 * i], boxes[6 * i + 1], boxes[6 * i + 2]);
        const V3 hi = v3(boxes[6 * i + 3], boxes[6 * i + 4], boxes[6 * i + 5]);
        BoxHits a{&with, lo, hi, {}}, b{&without, lo, hi, {}};
        mesh_query_aabb(with, lo, hi, a);
        mesh_query_aabb(without, lo, hi, b);
        if (a.t != b.t) return -1;
        *n_hits += (long)a.t.size();
        uint32_t begin, end;
        served += leaf_list(with.box_grid, lo, hi, begin, end) >= 0;
    }
    return served;
}

// The same over n rays (from, to).
int ll_rays(void* p, int n, const float* rays, long* n_hits) {
    const MeshView with = ((HostMesh*)p)->view();
    MeshView without = with;
    without.ray_grid.items = nullptr;
    int served = 0;
    for (int i = 0; i < n; i++) {
        const V3 from = v3(rays[6 * i], rays[6 * i + 1], rays[6 * i + 2]);
        const V3 to = v3(rays[6 * i + 3], rays[6 * i + 4], rays[6 * i + 5]);
        RayHits a{&with, from, to, 1.f, v3zero(), {}}, b{&without, from, to, 1.f, v3zero(), {}};
        mesh_query_ray(with, from, to, a);
        mesh_query_ray(without, from, to, b);
        if (a.t != b.t || std::memcmp(&a.frac, &b.frac, 4) != 0 || std::memcmp(&a.n, &b.n, 12) != 0) return -1;
        *n_hits += (long)a.t.size();
        const V3 rmin = v3(fminf(from.x, to.x), fminf(from.y, to.y), fminf(from.z, to.z));
        const V3 rmax = v3(fmaxf(from.x, to.x), fmaxf(from.y, to.y), fmaxf(from.z, to.z));
        uint32_t begin, end;
        served += leaf_list(with.ray_grid, rmin, rmax, begin, end) >= 0;
    }
    return served;
}

}  // extern "C"
