// rsg_mesh.h -- a shared, read-only arena collision mesh: triangles and a
// 16-bit quantized AABB tree over them.
//
// One copy lives in HBM for the whole batch (every arena uses the same
// mesh), so after the first ticks it is L2-resident.  The tree follows the
// published quantized-AABB-tree scheme the reference uses
// (BulletCollision/BroadphaseCollision/btQuantizedBvh.cpp:116-305,
// BulletCollision/CollisionShapes/btOptimizedBvh.cpp:28-188): leaves in
// triangle order, mean-split along the axis of largest centroid variance,
// depth-first node array with escape indices, 16-bit quantization with a 1 m
// margin, and subtree headers for trees larger than 2 KiB.  Traversal order is
// part of the contract: it decides the order contacts reach the solver.
#pragma once

#include "rsg_math.h"

namespace rsg {

struct QNode {
    uint16_t qmin[3];
    uint16_t qmax[3];
    int32_t esc_or_tri;  // >= 0: leaf, triangle index (part 0); < 0: -escape index
};

struct QSubtree {
    uint16_t qmin[3];
    uint16_t qmax[3];
    int32_t root;
    int32_t size;
};

constexpr int MAX_TRI_INFO_EDGES = 3;

// Per-triangle internal-edge data (btTriangleInfo, BulletCollision/CollisionShapes/btTriangleInfoMap.h:37-54).
struct TriInfo {
    float edge_angle[3];
    uint32_t flags;
};

// Broadphase grid of the reference arena (btRSBroadphase with
// ArenaConfig defaults, src/Sim/Arena/ArenaConfig/ArenaConfig.h:20-41):
// cell = 370 uu, bounds (-5600,-6000,0)..(5600,6000,2200) uu.
constexpr int BP_CELLS_X = 31, BP_CELLS_Y = 33, BP_CELLS_Z = 6;
constexpr int BP_NUM_CELLS = BP_CELLS_X * BP_CELLS_Y * BP_CELLS_Z;

// A triangle as the leaf lists hold it: its box (grown for ray lists), its
// index and its leaf node.
struct alignas(16) MeshLeaf {
    V3 lo;
    int32_t tri;
    V3 hi;
    int32_t node;
};

// Per-cell candidate lists on a uniform grid over the mesh: cell c's list
// holds, in the tree's visiting order, every leaf whose box touches the cell
// extended by `reach` towards +x, +y and +z.  A query box no larger than
// `reach` that starts in the cell therefore finds all its triangles in that
// one list, in the order the tree walk would reach them.  items may be null
// (no lists: walk the tree).
struct LeafGrid {
    const MeshLeaf* leaves;
    const uint32_t* items;    // indices into leaves
    const uint32_t* offsets;  // nx * ny * nz + 1
    int nx, ny, nz;
    V3 origin;
    float inv_cell, reach;
};

struct MeshView {
    const float* verts;      // 3 floats per vertex (Bullet units)
    const int32_t* tris;     // 3 indices per triangle
    const QNode* nodes;
    const QSubtree* subtrees;
    const TriInfo* tri_info; // may be null
    int n_tris, n_nodes, n_subtrees;
    V3 bvh_min, bvh_max, quant;
    V3 aabb_min, aabb_max;   // local AABB of the mesh (no margin)
    float tri_info_equal_vertex_threshold, tri_info_edge_distance_threshold,
          tri_info_convex_epsilon, tri_info_planar_epsilon, tri_info_max_edge_angle;
    // Occupancy bitmask on a uniform grid over the tree bounds: bit set iff a
    // triangle's box (grown by MESH_OCC_SLACK) touches the cell.  Lets a query
    // whose box touches no marked cell skip the tree walk (no triangle there
    // can yield a contact or a ray hit).  May be null.
    const uint32_t* occ;
    int occ_nx, occ_ny, occ_nz;
    V3 occ_origin;
    float occ_inv_cell;
    // Candidate lists of the box queries and of the wheel rays.
    LeafGrid box_grid, ray_grid;
};

constexpr float MESH_OCC_CELL = 2.f;     // Bullet units
constexpr float MESH_OCC_SLACK = 0.01f;
// Leaf lists: the ball's box (4.02 m in Hoops) and a car's (3.1 m) are within
// the box reach, a suspension ray (about 1.1 m) within the ray reach.
constexpr float LEAF_BOX_CELL = 2.f, LEAF_BOX_REACH = 4.25f;
constexpr float LEAF_RAY_CELL = 1.f, LEAF_RAY_REACH = 1.5f;

// True when no triangle of the mesh touches the box [lo, hi]: every grid
// cell the (slightly grown) box touches is unmarked.  Boxes touching many
// cells, or with non-finite bounds, report false (walk the tree).
RSG_FN bool mesh_region_empty(const MeshView& m, V3 lo, V3 hi) {
    if (!m.occ) return false;
    if (!(lo.x <= hi.x && lo.y <= hi.y && lo.z <= hi.z)) return false;
    V3 a = (lo - v3(MESH_OCC_SLACK, MESH_OCC_SLACK, MESH_OCC_SLACK) - m.occ_origin) * m.occ_inv_cell;
    V3 b = (hi + v3(MESH_OCC_SLACK, MESH_OCC_SLACK, MESH_OCC_SLACK) - m.occ_origin) * m.occ_inv_cell;
    if (!(fabsf(a.x) < 1e6f && fabsf(a.y) < 1e6f && fabsf(a.z) < 1e6f && fabsf(b.x) < 1e6f &&
          fabsf(b.y) < 1e6f && fabsf(b.z) < 1e6f))
        return false;
    int i0 = (int)floorf(a.x), j0 = (int)floorf(a.y), k0 = (int)floorf(a.z);
    int i1 = (int)floorf(b.x), j1 = (int)floorf(b.y), k1 = (int)floorf(b.z);
    i0 = i0 < 0 ? 0 : i0; j0 = j0 < 0 ? 0 : j0; k0 = k0 < 0 ? 0 : k0;
    i1 = i1 >= m.occ_nx ? m.occ_nx - 1 : i1;
    j1 = j1 >= m.occ_ny ? m.occ_ny - 1 : j1;
    k1 = k1 >= m.occ_nz ? m.occ_nz - 1 : k1;
    if (i0 > i1 || j0 > j1 || k0 > k1) return true;  // entirely outside the grid, which covers the mesh
    if ((i1 - i0 + 1) * (j1 - j0 + 1) * (k1 - k0 + 1) > 64) return false;
    for (int i = i0; i <= i1; i++)
        for (int j = j0; j <= j1; j++)
            for (int k = k0; k <= k1; k++) {
                int bit = (i * m.occ_ny + j) * m.occ_nz + k;
                if (m.occ[bit >> 5] >> (bit & 31) & 1u) return false;
            }
    return true;
}

RSG_FN void quantize(const MeshView& m, uint16_t out[3], V3 p, int is_max) {
    V3 v = (p - m.bvh_min) * m.quant;
    if (is_max) {
        out[0] = (uint16_t)(((uint16_t)(v.x + 1.f)) | 1);
        out[1] = (uint16_t)(((uint16_t)(v.y + 1.f)) | 1);
        out[2] = (uint16_t)(((uint16_t)(v.z + 1.f)) | 1);
    } else {
        out[0] = (uint16_t)(((uint16_t)(v.x)) & 0xfffe);
        out[1] = (uint16_t)(((uint16_t)(v.y)) & 0xfffe);
        out[2] = (uint16_t)(((uint16_t)(v.z)) & 0xfffe);
    }
}

RSG_FN void quantize_clamp(const MeshView& m, uint16_t out[3], V3 p, int is_max) {
    V3 c = p;
    c.x = c.x < m.bvh_min.x ? m.bvh_min.x : c.x;
    c.y = c.y < m.bvh_min.y ? m.bvh_min.y : c.y;
    c.z = c.z < m.bvh_min.z ? m.bvh_min.z : c.z;
    c.x = c.x > m.bvh_max.x ? m.bvh_max.x : c.x;
    c.y = c.y > m.bvh_max.y ? m.bvh_max.y : c.y;
    c.z = c.z > m.bvh_max.z ? m.bvh_max.z : c.z;
    quantize(m, out, c, is_max);
}

RSG_FN V3 unquantize(const MeshView& m, const uint16_t q[3]) {
    return v3((float)q[0] / m.quant.x, (float)q[1] / m.quant.y, (float)q[2] / m.quant.z) + m.bvh_min;
}

RSG_FN bool q_overlap(const uint16_t amin[3], const uint16_t amax[3], const uint16_t bmin[3], const uint16_t bmax[3]) {
    return !(amin[0] > bmax[0] || amax[0] < bmin[0] || amin[1] > bmax[1] || amax[1] < bmin[1] ||
             amin[2] > bmax[2] || amax[2] < bmin[2]);
}

RSG_FN void mesh_triangle(const MeshView& m, int t, V3 out[3]) {
    for (int j = 0; j < 3; j++) {
        int vi = m.tris[3 * t + j];
        out[j] = v3(m.verts[3 * vi], m.verts[3 * vi + 1], m.verts[3 * vi + 2]);
    }
}

// Cell list of a query box [lo, hi]: 1 and the list's range, 0 when no leaf
// can touch the box, -1 when the lists do not serve it (no lists, a box
// larger than their reach, non-finite bounds).
RSG_FN int leaf_list(const LeafGrid& g, V3 lo, V3 hi, uint32_t& begin, uint32_t& end) {
    if (!g.items) return -1;
    const V3 d = hi - lo;
    if (!(d.x >= 0.f && d.y >= 0.f && d.z >= 0.f && d.x <= g.reach && d.y <= g.reach && d.z <= g.reach)) return -1;
    const V3 f = (lo - g.origin) * g.inv_cell;
    if (!(fabsf(f.x) < 1e6f && fabsf(f.y) < 1e6f && fabsf(f.z) < 1e6f)) return -1;
    int i = (int)f.x, j = (int)f.y, k = (int)f.z;
    if (i >= g.nx || j >= g.ny || k >= g.nz) return 0;  // past the grid, which covers the mesh
    i = i < 0 ? 0 : i; j = j < 0 ? 0 : j; k = k < 0 ? 0 : k;
    const int c = (i * g.ny + j) * g.nz + k;
    begin = g.offsets[c];
    end = g.offsets[c + 1];
    return begin < end ? 1 : 0;
}

RSG_FN bool boxes_touch(V3 alo, V3 ahi, V3 blo, V3 bhi) {
    return alo.x <= bhi.x && ahi.x >= blo.x && alo.y <= bhi.y && ahi.y >= blo.y && alo.z <= bhi.z && ahi.z >= blo.z;
}

// Leaves of list items [at, at + 4) below `end` whose box touches [lo, hi]
// (bit r: item at + r).  The four loads are independent, so they overlap.
RSG_FN uint32_t leaf_list_mask(const LeafGrid& g, uint32_t at, uint32_t end, V3 lo, V3 hi, MeshLeaf leaf[4]) {
    uint32_t idx[4];
    for (int r = 0; r < 4; r++) idx[r] = g.items[at + r < end ? at + r : at];
    for (int r = 0; r < 4; r++) leaf[r] = g.leaves[idx[r]];
    uint32_t m = 0;
    for (int r = 0; r < 4; r++)
        if (at + r < end && boxes_touch(leaf[r].lo, leaf[r].hi, lo, hi)) m |= 1u << r;
    return m;
}

// AABB query in the reference's order (walkStacklessQuantizedTreeCacheFriendly,
// btQuantizedBvh.cpp:605-625 -> walkStacklessQuantizedTree :627-665).
// cb(int tri) is called for every leaf whose box overlaps: by the cell's list
// exactly those whose triangle's box does, by the tree also some whose
// quantized box does (callers test the triangle's box themselves; a
// triangle's quantized box contains it, so none is missed).
template <class CB>
RSG_FN void mesh_query_aabb(const MeshView& m, V3 qmin_f, V3 qmax_f, CB& cb) {
    uint32_t at, end;
    const int listed = leaf_list(m.box_grid, qmin_f, qmax_f, at, end);
    if (listed == 0) return;
    if (listed > 0) {
        for (; at < end; at += 4) {
            MeshLeaf leaf[4];
            uint32_t mask = leaf_list_mask(m.box_grid, at, end, qmin_f, qmax_f, leaf);
            while (mask) {
                const int t = pick(__builtin_ctz(mask), leaf[0].tri, leaf[1].tri, leaf[2].tri, leaf[3].tri);
                mask &= mask - 1u;
                cb(t);
            }
        }
        return;
    }
    if (mesh_region_empty(m, qmin_f, qmax_f)) return;
    uint16_t qmin[3], qmax[3];
    quantize_clamp(m, qmin, qmin_f, 0);
    quantize_clamp(m, qmax, qmax_f, 1);
    for (int s = 0; s < m.n_subtrees; s++) {
        const QSubtree& st = m.subtrees[s];
        if (!q_overlap(qmin, qmax, st.qmin, st.qmax)) continue;
        int cur = st.root, end_node = st.root + st.size;
        while (cur < end_node) {
            const QNode& n = m.nodes[cur];
            bool ov = q_overlap(qmin, qmax, n.qmin, n.qmax);
            bool leaf = n.esc_or_tri >= 0;
            if (leaf && ov) cb(n.esc_or_tri);
            if (ov || leaf) cur++;
            else cur += -n.esc_or_tri;
        }
    }
}

// A ray as the tree's box test takes it (LinearMath/btAabbUtil2.h:82-115).
struct TreeRay {
    V3 from, inv;
    float lambda_max;
    uint16_t qmin[3], qmax[3];
};

// Whether the walk descends into (or, at a leaf, reports) node n.  A parent's
// box contains its children's and the test is monotone in the box, so a leaf
// that passes is one the walk reaches.
RSG_FN bool ray_meets_node(const MeshView& m, const QNode& n, const TreeRay& r) {
    if (!q_overlap(r.qmin, r.qmax, n.qmin, n.qmax)) return false;
    const V3 lo = unquantize(m, n.qmin), hi = unquantize(m, n.qmax);
    const bool nx = r.inv.x < 0.f, ny = r.inv.y < 0.f, nz = r.inv.z < 0.f;
    float tmin = ((nx ? hi.x : lo.x) - r.from.x) * r.inv.x;
    float tmax = ((nx ? lo.x : hi.x) - r.from.x) * r.inv.x;
    const float tymin = ((ny ? hi.y : lo.y) - r.from.y) * r.inv.y;
    const float tymax = ((ny ? lo.y : hi.y) - r.from.y) * r.inv.y;
    if ((tmin > tymax) || (tymin > tmax)) return false;
    if (tymin > tmin) tmin = tymin;
    if (tymax < tmax) tmax = tymax;
    const float tzmin = ((nz ? hi.z : lo.z) - r.from.z) * r.inv.z;
    const float tzmax = ((nz ? lo.z : hi.z) - r.from.z) * r.inv.z;
    if ((tmin > tzmax) || (tzmin > tmax)) return false;
    if (tzmin > tmin) tmin = tzmin;
    if (tzmax < tmax) tmax = tzmax;
    return (tmin < r.lambda_max) && (tmax > 0.f);
}

// Ray query (walkStacklessQuantizedTreeAgainstRay with RAYAABB2,
// btQuantizedBvh.cpp:531-603 and LinearMath/btAabbUtil2.h:82-115).
template <class CB>
RSG_FN void mesh_query_ray(const MeshView& m, V3 from, V3 to, CB& cb) {
    const V3 rmin = v3(fminf(from.x, to.x), fminf(from.y, to.y), fminf(from.z, to.z));
    const V3 rmax = v3(fmaxf(from.x, to.x), fmaxf(from.y, to.y), fmaxf(from.z, to.z));
    uint32_t at = 0, end = 0;
    const int listed = leaf_list(m.ray_grid, rmin, rmax, at, end);
    if (listed == 0 || (listed < 0 && mesh_region_empty(m, rmin, rmax))) return;
    TreeRay r;
    const V3 dir = safe_normalized(to - from);
    r.from = from;
    r.lambda_max = dot(dir, to - from);
    r.inv = v3(dir.x == 0.f ? 1e18f : 1.f / dir.x, dir.y == 0.f ? 1e18f : 1.f / dir.y,
               dir.z == 0.f ? 1e18f : 1.f / dir.z);
    quantize_clamp(m, r.qmin, rmin, 0);
    quantize_clamp(m, r.qmax, rmax, 1);
    if (listed > 0) {
        for (; at < end; at += 4) {
            MeshLeaf leaf[4];
            uint32_t mask = leaf_list_mask(m.ray_grid, at, end, rmin, rmax, leaf);
            while (mask) {
                const int r4 = __builtin_ctz(mask);
                const int t = pick(r4, leaf[0].tri, leaf[1].tri, leaf[2].tri, leaf[3].tri);
                const int node = pick(r4, leaf[0].node, leaf[1].node, leaf[2].node, leaf[3].node);
                mask &= mask - 1u;
                if (ray_meets_node(m, m.nodes[node], r)) cb(t);
            }
        }
        return;
    }
    int cur = 0;
    while (cur < m.n_nodes) {
        const QNode& n = m.nodes[cur];
        const bool ray_ov = ray_meets_node(m, n, r);
        const bool leaf = n.esc_or_tri >= 0;
        if (leaf && ray_ov) cb(n.esc_or_tri);
        if (ray_ov || leaf) cur++;
        else cur += -n.esc_or_tri;
    }
}

}  // namespace rsg
