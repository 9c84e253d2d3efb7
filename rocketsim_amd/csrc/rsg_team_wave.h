// rsg_team_wave.h -- the parts of the team tick (rsg_team.h) that all teams of
// a wave run together, for the cooperative step kernel and the ball-prediction
// kernel.  Device code only.
#pragma once

#include "rsg_team.h"

namespace rsg {

// Narrowphase of every arena of the wave: `team()` gives this lane's team, `on`
// whether it takes part.  The rounds run for all teams together; a search that
// needs the penetration pass gets the wave's one work space `small` in turn.
//
// What bounds it: the searches, each a chain of dependent loads and
// arithmetic.  One lane went through a manifold's triangles before, 2 to 10 us
// each, and ran the whole pair again for a penetration (2v2 x 4096 arenas 0.272
// ms a tick against 0.194, as a wave waits for its slowest; a ball rolling on
// the mesh 30 us a tick against 12).
template <class MakeTeam>
__device__ __forceinline__ void team_narrow(MakeTeam&& team, bool on, EpaSmall* small, uint64_t team_mask) {
    if (on) team().narrow(0);
    __syncthreads();
    {
        Team t = team();
        const int self = (int)threadIdx.x;
        Team::Search search;
        search.more = on;
        bool first = true;
        RSG_UNROLL_1
        while (__any(search.more)) {
            int tri = -1, mi = -1;
            if (search.more) mi = t.next_search(search, first, tri);
            first = false;
            V3 n, pb;
            float dist = 0.f;
            int found = 0;
            uint64_t waiting = 0;
            // once without the penetration pass, then those that need it in turn
            RSG_UNROLL_1
            for (int turn = 0; turn == 0 || waiting; turn++) {
                if (turn == 0 ? mi >= 0 : self == __builtin_ctzll(waiting)) {
                    const EpaWork w0 = epa_work(*small), w1 = epa_work(t.g->epa);
                    found = t.contact(search.q, mi, tri, turn ? &w0 : nullptr, &w1, n, pb, dist);
                }
                __syncthreads();
                waiting = turn == 0 ? __ballot(found < 0) : waiting & (waiting - 1u);
            }
            // into the manifolds, each team's lanes in order
            uint64_t left = __ballot(found > 0) & team_mask;
            RSG_UNROLL_1
            while (__any(left != 0)) {
                if (left && self == __builtin_ctzll(left))
                    t.add_point(mi, search.q, n, pb, dist, false, tri >= 0 ? t.mesh_of(mi) : nullptr, tri);
                __syncthreads();
                left &= left - 1u;
            }
        }
    }
    __syncthreads();
    if (on) team().refresh_all();
    __syncthreads();
    if (on) team().narrow(1);
    __syncthreads();
}

// The levels (rows() in rsg_team.h) on which any of the wave's lanes with `in`
// has its row, one bit each; bit 63 stands for all from there on.
__device__ __forceinline__ uint64_t wave_levels(bool in, int level) {
    uint64_t levels = 0;
    for (uint64_t m = __ballot(in); m; m &= m - 1u) {
        const int lv = __builtin_amdgcn_readlane(level, __builtin_ctzll(m));
        levels |= 1ull << (lv < 63 ? lv : 63);
    }
    return levels;
}

// Solver of every arena of the wave (Team::row_visit's passes): contact r of
// an arena on its lane r, both rows in registers; an arena with more contacts
// than lanes keeps its rows in global memory.  One loop runs the split-impulse
// passes, then contact and friction rows in turn, level by level, so that a
// row's update is in the code once.
//
// What bounds it: a chain of row updates through LDS, 0.3 us each.  A pass
// goes only over the levels that have rows acting in it (a ball on the arena's
// mesh has a row for each triangle, of which the averaged one alone acts after
// the split passes), and an arena whose contact and friction rows all end an
// iteration as they began it is done: the iterations left would repeat it.
__device__ __forceinline__ void team_solve(Team& t, bool live, float dt, uint64_t team_mask) {
    const int n = live ? t.h->n_rows : 0, levels = live ? t.h->n_levels : 0;
    if (!__any(n > 0)) return;
    const bool in_memory = n > t.lanes;
    TeamRow row;
    int level = -1;
    bool splits = false, acts = false;
    RSG_UNROLL_1
    for (int r = t.lane; r < n; r += t.lanes) {
        t.row_setup(r, dt, row);
        level = t.h->row.level[r];
        splits = row.c.rhs_pen != 0.f;
        acts = !row.c.special;
        if (in_memory) t.g->rows[r] = row;
    }
    uint64_t split_levels, contact_levels;
    if (__any(in_memory)) {
        split_levels = contact_levels = ~0ull;
    } else {
        split_levels = wave_levels(splits, level);
        contact_levels = wave_levels(acts, level);
    }
    int what = split_levels ? 0 : 1, it = 0;
    bool go = n > 0, moved = false;
    RSG_UNROLL_1
    while (true) {
        RSG_UNROLL_1
        for (uint64_t todo = what == 0 ? split_levels : contact_levels; todo; todo &= todo - 1u) {
            int lv = __builtin_ctzll(todo);
            if (!__any(go && lv < levels)) break;
            RSG_UNROLL_1
            do {  // once, but for all levels from 63 on
                if (go) {
                    RSG_UNROLL_1
                    for (int r = t.lane; r < n; r += t.lanes) {
                        if ((in_memory ? (int)t.h->row.level[r] : level) != lv) continue;
                        if (in_memory) row = t.g->rows[r];
                        const float q = t.row_visit(row, what);
                        moved |= what == 0 ? !(q * q <= 0.f) : q != 0.f;
                        if (in_memory) t.g->rows[r] = row;
                    }
                }
                __syncthreads();
                lv++;
            } while (lv > 63 && __any(go && lv < levels));
        }
        if (what == 1) {
            what = 2;
            continue;
        }
        // an arena's passes of either kind end once one moves nothing
        go = go && (__ballot(moved) & team_mask) != 0;
        moved = false;
        if (++it < SOLVER_ITERATIONS && __any(go)) {
            what = what == 0 ? 0 : 1;
        } else if (what == 0) {
            what = 1;
            it = 0;
            go = n > 0;
        } else {
            break;
        }
    }
}

}  // namespace rsg
