// rsg_team.h -- one arena's tick (Arena::Step, src/Sim/Arena/Arena.cpp:689-756)
// by a team of lanes, in phases with a barrier between them: the cooperative
// step kernel and the ball-prediction kernel run these.  A phase is a function
// of the lane; lanes exchange data only from one phase to the next, through
// the team's local block (LDS on the device), so the host can run a phase lane
// by lane (tests/cpp/team_host.cpp does, against arena_tick).
//
// Phases of a tick (results are those of arena_tick, bit for bit):
//   begin        controls, one car per lane; the ball's sleep flag
//   rays         one wheel per lane
//   car_begin    one car per lane   \  all cars at once, or one after another in
//   wheels       one wheel per lane  > the update order when a wheel rests on a
//   car          one car per lane   /  car or a car respawns
//   body_begin   one body per lane: gravity, damping, proxy AABB, cell
//   ranks, pairs, plan   one body per lane: broadphase order, its pairs, their
//                manifolds
//   narrow 0     one manifold per lane: planes, two cars
//   search       in rounds: the cars' contacts with the ball, then each mesh
//                manifold's triangles, one a lane; the points go in in lane order,
//                their callbacks' effects recorded
//   refresh_all  one manifold per lane
//   narrow 1     lane 0, in pair order: the effects (pairs with more than fit the
//                record run again here)
//   rows         lane 0: islands, the contact rows and their levels
//   solve        one contact (its normal and friction row) per lane
//   body_end     one body per lane: write-back, integration, post-tick
//   pads         pads spread over the lanes
//   end          lane 0: pad pickups, goal test
//
// What bounds it: latency, not issue or bandwidth.  The phases replaced a
// kernel whose serial lane did most of this through global work space: 839 KB
// of code against an instruction cache of 64 KB, 3.4 KB of private memory per
// lane and 1600 vector memory operations a wave-tick.  Here every algorithm
// has one inlined instance, the working set of an ordinary tick is in LDS and
// registers (185 vector reads a wave-tick), and what is rare (penetration,
// box-box, kickoff) is out of line.  2v2 x 16384 arenas: 0.350 ms a tick against
// 0.863; one 1v1 arena: 0.031 against 0.059.  Waves still wait 47 % of their
// time, and a launch ends with its slowest wave.
#pragma once

#include "rsg_tick.h"

namespace rsg {

// Manifolds kept in the local block; an arena has 2-4 in ordinary play (97 %
// of the ticks of 2v2 melees have at most 5), the rest go to global memory.
constexpr int TEAM_LOCAL_MF = 5;

// A contact point before the solver: what a manifold needs to keep, replace
// and refresh it.  World points and material follow from these.
struct TeamPoint {
    V3 la, lb, n;
    float dist;
};
struct TeamManifold {
    float threshold, friction, restitution;
    uint8_t n;
    uint8_t special;   // ball against the world: solved through the averaged row
    uint8_t n_effects;
    uint8_t redo;      // run again in order (two cars, effects past the record)
    TeamPoint p[MAX_POINTS_PER_MANIFOLD];
    int eff_code;      // the first effect (kind | car a << 8), unless car-car
    V3 eff_v;
};

// A wheel's results: its ray, then what the car's logic needs of it.
struct TeamWheel {
    union {
        RayHit hit;
        struct {
            V3 normal;
            V3 sus_v, sus_w, tire_v, tire_w;  // velocity changes of its two impulses
            uint32_t flags;
        } out;
    };
};
enum { TW_CONTACT = 1u, TW_WORLD = 2u, TW_SUS = 4u, TW_TIRE = 8u };

struct TeamBody {
    V3 amin, amax;                // proxy AABB
    V3 dv, dw, push, turn;        // solver velocities
    uint32_t statics, statics_kept;    // overlapped statics; those with a manifold
    uint16_t dyn, dyn_made, dyn_kept;  // the same for later bodies, by broadphase rank
    uint16_t pad_window;          // cars: pad grid cells within reach (x0 | x1 << 4 | y0 << 8 | y1 << 12)
    int cell;                     // broadphase cell of this tick
    uint32_t rank;                // place in the cell lists' order
};

constexpr uint16_t TEAM_NO_PADS = 0x000fu;  // x0 = 15, x1 = 0: no window

struct TeamHead {
    int n_mf, n_rows, n_levels;
    uint8_t respawn[RSG_MAX_CARS];        // car respawns this tick
    uint8_t on_car[4 * RSG_MAX_CARS];     // wheel rests on a car
    uint8_t order[MAX_BODIES];            // bodies by broadphase rank
    uint8_t overflow[MAX_BODIES];         // RSG_STATUS_* found by a body's lane
    uint8_t any_locked;
    int8_t mf_b0[MAX_MANIFOLDS], mf_b1[MAX_MANIFOLDS];
    uint8_t im[MAX_MANIFOLDS];            // island manifolds, sorted
    union {
        struct { uint8_t key[MAX_MANIFOLDS], lo[MAX_MANIFOLDS], hi[MAX_MANIFOLDS]; } sort;
        struct { uint8_t src[MAX_ROWS], level[MAX_ROWS]; } row;  // manifold | point << 6, or 255: the special row
    };
    // the ball's averaged world contact (SpecialInfo)
    int sp_num;
    float sp_friction, sp_restitution, sp_dist;
    V3 sp_normal;
};
constexpr uint8_t ROW_SPECIAL = 255;

// One contact's two rows.
struct TeamRow {
    SRow c, f;
    int a, b;          // body codes
};

// An arena's block of global memory: what does not fit the local block.
struct TeamGlobal {
    TeamManifold mf[MAX_MANIFOLDS];
    TeamRow rows[MAX_ROWS];
    EpaSpace epa;
    PairLog log;
};
static_assert(sizeof(TeamGlobal) <= sizeof(ArenaSpace), "the team's global block must fit the arena's");

// Bytes of the local block after the arena itself, for `lanes` lanes (4 per
// car slot): the head, then the wheels' results or the world step's tables.
RSG_FN size_t team_local_bytes(int max_cars) {
    const size_t wheels = (size_t)(4 * max_cars) * sizeof(TeamWheel);
    const size_t world = (size_t)(1 + max_cars) * sizeof(TeamBody) + TEAM_LOCAL_MF * sizeof(TeamManifold);
    return sizeof(TeamHead) + (wheels > world ? wheels : world);
}

// Effects out of line: rarely more than a flag, and long.
RSG_COLD_FN void team_apply_effect(ArenaLocal& A, int code, V3 v0, V3 v1) {
    World w(A, nullptr, false);
    w.apply_effect(code & 0xff, (code >> 8) & 0xff, code >> 16, v0, v1);
}
RSG_COLD_FN void team_kickoff(ArenaLocal& A, uint64_t seed, uint32_t arena_id) { arena_kickoff_reset(A, seed, arena_id); }

// The triangles a box meets (mesh_query_aabb), handed to a team's lanes: of a
// leaf list one item a lane and round, of the tree, which serves what the lists
// do not, one a round to lane 0 (every lane walks it).  The order of the query's report is that of
// the rounds, and of the lanes within a round.
struct MeshBoxIter {
    const MeshView* m;
    V3 lo, hi;
    int mode;            // 0: done, 1: leaf list, 2: tree
    uint32_t at, end;
    uint16_t qmin[3], qmax[3];
    int sub, cur, cur_end;

    RSG_FN void start(const MeshView* mesh, V3 l, V3 h) {
        m = mesh; lo = l; hi = h;
        at = end = 0;
        mode = 0;
        const int listed = leaf_list(m->box_grid, lo, hi, at, end);
        if (listed == 0) return;
        if (listed > 0) { mode = 1; return; }
        if (mesh_region_empty(*m, lo, hi)) return;
        mode = 2;
        quantize_clamp(*m, qmin, lo, 0);
        quantize_clamp(*m, qmax, hi, 1);
        sub = -1;
        cur = cur_end = 0;
    }
    // This lane's triangle of the round, or -1; mode 0 after the last round.
    RSG_FN int next(int lane, int lanes) {
        if (mode == 1) {
            int tri = -1;
            if (at + (uint32_t)lane < end) {
                const MeshLeaf leaf = m->box_grid.leaves[m->box_grid.items[at + (uint32_t)lane]];
                if (boxes_touch(leaf.lo, leaf.hi, lo, hi)) tri = leaf.tri;
            }
            at += (uint32_t)lanes;
            if (at >= end) mode = 0;
            return tri;
        }
        if (mode == 0) return -1;
        while (true) {
            while (cur >= cur_end) {
                if (++sub >= m->n_subtrees) { mode = 0; return -1; }
                const QSubtree& st = m->subtrees[sub];
                if (!q_overlap(qmin, qmax, st.qmin, st.qmax)) continue;
                cur = st.root;
                cur_end = st.root + st.size;
            }
            const QNode& n = m->nodes[cur];
            const bool ov = q_overlap(qmin, qmax, n.qmin, n.qmax), leaf = n.esc_or_tri >= 0;
            cur += ov || leaf ? 1 : -n.esc_or_tri;
            if (leaf && ov) return lane == 0 ? n.esc_or_tri : -1;
        }
    }
};

// Body 0's side of a manifold, and what the contacts of the pair need.
struct TeamPair {
    int b0;
    float thr, ball_r;
    bool respond;
    Xf x0, cx;        // the body's, its box's frame
    V3 he;            // half extents of the box with its margin
    V3 amin, amax;
};

struct Team {
    ArenaLocal& A;
    const ArenaGeom* geo;   // null without an arena
    TeamHead* h;
    TeamWheel* wheel;       // shares its place with body and lmf: used before the world step only
    TeamBody* body;
    TeamManifold* lmf;
    TeamGlobal* g;
    int lane, lanes;
    World w;                // geometry queries only

    RSG_FN Team(ArenaLocal& a, const ArenaGeom* ge, unsigned char* local, int max_cars, TeamGlobal* gl, int ln, int lns)
        : A(a), geo(ge), g(gl), lane(ln), lanes(lns), w(a, ge, ge != nullptr) {
        h = reinterpret_cast<TeamHead*>(local);
        unsigned char* u = local + sizeof(TeamHead);
        wheel = reinterpret_cast<TeamWheel*>(u);
        body = reinterpret_cast<TeamBody*>(u);
        lmf = reinterpret_cast<TeamManifold*>(u + (size_t)(1 + max_cars) * sizeof(TeamBody));
    }
    RSG_FN int bodies() const { return 1 + A.n_cars; }
    RSG_FN TeamManifold& manifold(int mi) { return mi < TEAM_LOCAL_MF ? lmf[mi] : g->mf[mi]; }

    // -----------------------------------------------------------------------
    // Cars

    RSG_FN void begin(const TickParams& P) {
        if (lane < A.n_cars) {
            tick_car_controls(A, P, lane);
            const Car& c = A.cars[lane];
            h->respawn[lane] = flag(c.flags, RSG_CF_DEMOED) && rs_max(c.demo_timer - P.dt, 0.f) == 0.f;
        }
        if (lane == 0) tick_ball_sleep(A);
    }
    RSG_FN bool any_respawn() const {
        bool any = false;
        for (int i = 0; i < A.n_cars; i++) any |= h->respawn[i] != 0;
        return any;
    }
    // Pass -1: every wheel's ray at the start of the tick (no car respawns).
    // Pass p: the rays of the p-th car as the reference casts them in its turn
    // (a car respawned this tick: earlier cars have moved).
    RSG_FN void rays(int pass) {
        const int ci = lane >> 2;
        if (ci >= A.n_cars || (pass >= 0 && A.order[pass] != ci)) return;
        int pos = -1;
        if (pass < 0) {
            pos = 0;
            while (pos < A.n_cars && A.order[pos] != ci) pos++;
        }
        w.ray_caster_pos = pos;
        V3 source, target;
        wheel_ray(A.cars[ci], *A.cars[ci].phys, lane & 3, source, target);
        const RayHit r = w.raycast(source, target, 1 + ci);
        wheel[lane].hit = r;
        h->on_car[lane] = r.hit && !r.is_static && r.body >= 1;
    }
    // Whether the cars' updates do not depend on each other.
    RSG_FN bool independent() const {
        bool any = any_respawn();
        for (int i = 0; i < 4 * A.n_cars; i++) any |= h->on_car[i] != 0;
        return !any;
    }
    // Passes over the cars: all at once, or one by one in the update order.
    RSG_FN int car_passes(bool together) const { return together ? 1 : A.n_cars; }
    RSG_FN bool in_pass(bool together, int pass, int ci) const { return together || A.order[pass] == ci; }

    RSG_FN void car_begin(const TickParams& P, bool together, int pass) {
        if (lane < A.n_cars && in_pass(together, pass, lane)) car_pre_begin(A, P, lane);
    }
    RSG_FN void wheels(const TickParams& P, bool together, int pass) {
        if (lane >= 4 * A.n_cars || !in_pass(together, pass, lane >> 2)) return;
        const int i = lane & 3;
        Car& c = A.cars[lane >> 2];
        if (flag(c.flags, RSG_CF_DEMOED)) return;
        const CarPhys& cp = *c.phys;
        const float dt = P.dt;
        WheelT t;
        wheel_update_transform(c, cp, i, t);
        const RayHit hit = wheel[lane].hit;
        wheel_contact(c, t, cp, i, hit, A.si);
        wheel_friction_impulse(c, t, i, t.ground >= 0 ? w.body_ptr(t.ground) : nullptr, dt);
        wheel_update_friction(c, t, cp, i, car_next_handbrake(c, dt), car_real_throttle(c));
        wheel_susp_force(t, cp, i);
        auto& o = wheel[lane].out;
        uint32_t fl = (t.in_contact ? TW_CONTACT : 0u) | (t.with_world ? TW_WORLD : 0u);
        o.normal = t.contact_normal;
        V3 imp, rel;
        if (t.susp_force != 0) {
            fl |= TW_SUS;
            wheel_susp_impulse(c, t, i, dt, imp, rel);
            o.sus_v = imp * c.b.inv_mass;
            o.sus_w = c.b.inv_iw * cross(rel, imp);
        }
        if (!is_zero(t.impulse)) {
            fl |= TW_TIRE;
            wheel_tire_impulse(c, t, dt, imp, rel);
            o.tire_v = imp * c.b.inv_mass;
            o.tire_w = c.b.inv_iw * cross(rel, imp);
        }
        o.flags = fl;
    }
    RSG_FN void car(const TickParams& P, bool together, int pass) {
        if (lane >= A.n_cars || !in_pass(together, pass, lane)) return;
        Car& c = A.cars[lane];
        if (flag(c.flags, RSG_CF_DEMOED)) return;
        uint32_t contact = 0;
        bool on_world = false;
        V3 normal_sum = v3zero();
        for (int i = 0; i < 4; i++) {
            const auto& o = wheel[4 * lane + i].out;
            on_world |= (o.flags & TW_WORLD) != 0;
            if (!(o.flags & TW_CONTACT)) continue;
            contact |= 1u << i;
            normal_sum += o.normal;
        }
        car_pre_logic(A, P, c, contact, on_world, normal_sum);
        // vehicle_second's impulses: their velocity changes do not depend on
        // the velocity, so the wheels' lanes have computed them
        if (c.b.inv_mass != 0.f) {
            for (int i = 0; i < 4; i++) {
                const auto& o = wheel[4 * lane + i].out;
                if (o.flags & TW_SUS) { c.b.vel += o.sus_v; c.b.ang += o.sus_w; }
            }
            for (int i = 0; i < 4; i++) {
                const auto& o = wheel[4 * lane + i].out;
                if (o.flags & TW_TIRE) { c.b.vel += o.tire_v; c.b.ang += o.tire_w; }
            }
        }
        car_update_boost(c, P.dt, A.mut);
    }

    // -----------------------------------------------------------------------
    // Broadphase

    RSG_FN void body_begin(const TickParams& P) {
        if (lane >= bodies()) return;
        Body& b = *w.body_ptr(lane);
        if (lane == 0) ball_pre_tick(A.ball, P.mode, P.dt);
        if (b.active) b.force += b.grav;
        if (lane == 0) world_ball_damping(A, P.dt);
        TeamBody& t = body[lane];
        w.proxy_aabb(lane, P.dt, t.amin, t.amax);
        t.cell = bp_cell_of(t.amin);
        t.dv = t.dw = t.push = t.turn = v3zero();
    }
    // btRSBroadphase::setAabb: a proxy whose cell changed moves to the end of
    // the cell lists, the changed ones in index order.
    RSG_FN void ranks() {
        const int nb = bodies();
        if (lane >= nb) return;
        const bool mine = nb > 1 && body[lane].cell != A.bp_cell[lane];
        uint32_t r = 0;
        for (int j = 0; j < nb; j++) {
            const bool moved = nb > 1 && body[j].cell != A.bp_cell[j];
            bool before;
            if (moved != mine) before = mine;
            else if (moved) before = j < lane;
            else before = A.bp_seq[j] < A.bp_seq[lane] || (A.bp_seq[j] == A.bp_seq[lane] && j < lane);
            r += before ? 1u : 0u;
        }
        body[lane].rank = r;
        h->order[r] = (uint8_t)lane;
        h->overflow[lane] = 0;
    }
    // The body's overlapping pairs (statics, then the later bodies in list
    // order) and what the dispatcher does with each (World::plan_pairs).
    RSG_FN void pairs() {
        const int nb = bodies(), p = lane;
        if (p >= nb) return;
        TeamBody& t = body[p];
        A.bp_cell[p] = t.cell;
        A.bp_seq[p] = t.rank;
        const V3 amin = t.amin, amax = t.amax;
        V3 cmin = v3zero(), cmax = v3zero();
        if (p > 0) w.car_child_aabb(p, cmin, cmax);
        const bool awake = w.active(p);
        uint32_t st = 0, kept = 0;
        if (geo) {
            uint32_t cand = geo->cell_statics[t.cell];
            if (p > 0) cand &= ~geo->car_skip;
            const int ns = num_statics(*geo);
            for (int s = 0; s < ns; s++) {
                if (!(cand >> s & 1u)) continue;
                V3 smin, smax;
                static_shape_aabb(geo, s, smin, smax);
                const V3 th = v3(CONTACT_BREAKING_THRESHOLD, CONTACT_BREAKING_THRESHOLD, CONTACT_BREAKING_THRESHOLD);
                if (!aabb_overlap(amin, amax, smin - th, smax + th)) continue;
                st |= 1u << s;
                if (awake && (p == 0 || aabb_overlap(cmin, cmax, smin, smax))) kept |= 1u << s;
            }
        }
        uint32_t dyn = 0, made = 0, dkept = 0;
        for (int r = 0; r < nb; r++) {
            const int q = h->order[r];
            if (q <= p || !bp_cells_adjacent(body[q].cell, t.cell)) continue;
            if (!aabb_overlap(amin, amax, body[q].amin, body[q].amax)) continue;
            dyn |= 1u << r;
            if (!(awake || w.active(q))) continue;
            V3 qmin, qmax;
            w.car_child_aabb(q, qmin, qmax);
            bool creates = true, keeps;
            if (p == 0) {
                const float rad = make_ball_phys(A.ball.radius_uu, A.ball.mass).radius + 0.08f;
                const V3 e = v3(rad, rad, rad);
                creates = keeps = aabb_overlap(qmin, qmax, A.ball.b.pos - e, A.ball.b.pos + e);
            } else {
                V3 bmin, bmax;
                w.shape_aabb(q, A.cars[q - 1].b.pos, A.cars[q - 1].b.rot, bmin, bmax);
                keeps = aabb_overlap(cmin, cmax, bmin, bmax) && aabb_overlap(qmin, qmax, cmin, cmax);
            }
            if (creates) made |= 1u << r;
            if (keeps) dkept |= 1u << r;
        }
        t.statics = st;
        t.statics_kept = kept;
        t.dyn = (uint16_t)dyn;
        t.dyn_made = (uint16_t)made;
        t.dyn_kept = (uint16_t)dkept;
    }
    // Pairs past the capacity are dropped, the last ones first.
    RSG_FN void trim() {
        const int nb = bodies();
        if (lane >= nb) return;
        int before = 0;
        for (int p = 0; p < lane; p++) before += pop(body[p].statics) + pop(body[p].dyn);
        TeamBody& t = body[lane];
        const int mine = pop(t.statics) + pop(t.dyn);
        int drop = before + mine - MAX_PAIRS;
        if (drop > mine) drop = mine;
        if (drop <= 0) return;
        // noted for the later phases; the masks change in plan(), once every lane has counted
        h->overflow[lane] = (uint8_t)drop;
    }
    RSG_FN static int pop(uint32_t x) { return __builtin_popcount(x); }
    RSG_FN static uint32_t top_bit(uint32_t x) { return 1u << (31 - __builtin_clz(x)); }
    RSG_FN void drop_pairs() {
        if (lane >= bodies()) return;
        TeamBody& t = body[lane];
        int drop = h->overflow[lane];
        h->overflow[lane] = drop ? RSG_STATUS_CONTACT_OVERFLOW : 0;
        for (; drop > 0; drop--) {
            if (t.dyn) {
                const uint16_t keep = (uint16_t)~top_bit(t.dyn);
                t.dyn &= keep; t.dyn_made &= keep; t.dyn_kept &= keep;
            } else {
                const uint32_t keep = ~top_bit(t.statics);
                t.statics &= keep; t.statics_kept &= keep;
            }
        }
    }
    // The manifolds, numbered in pair order.
    RSG_FN void plan() {
        const int nb = bodies(), p = lane;
        if (p >= nb) return;
        int n = 0;
        for (int q = 0; q < p; q++) n += pop(body[q].statics_kept) + pop(body[q].dyn_kept);
        const TeamBody& t = body[p];
        const int mine = pop(t.statics_kept) + pop(t.dyn_kept);
        if (p == nb - 1) h->n_mf = n + mine < MAX_MANIFOLDS ? n + mine : MAX_MANIFOLDS;
        if (p == 0) h->any_locked = 0;
        if (n + mine < MAX_MANIFOLDS) {
            for (uint32_t m = t.statics_kept; m; m &= m - 1u) {
                h->mf_b0[n] = (int8_t)p;
                h->mf_b1[n] = (int8_t)(-1 - __builtin_ctz(m));
                n++;
            }
            for (uint32_t m = t.dyn_kept; m; m &= m - 1u) {
                h->mf_b0[n] = (int8_t)h->order[__builtin_ctz(m)];
                h->mf_b1[n] = (int8_t)p;
                n++;
            }
            return;
        }
        // the capacity is reached at this body: a pair that makes a manifold
        // past it is flagged and dropped
        const uint32_t st_made = w.active(p) ? t.statics : 0u;
        bool over = false;
        for (uint32_t m = st_made; m; m &= m - 1u) {
            const int s = __builtin_ctz(m);
            if (n >= MAX_MANIFOLDS) { over = true; continue; }
            if (!(t.statics_kept >> s & 1u)) continue;
            h->mf_b0[n] = (int8_t)p;
            h->mf_b1[n] = (int8_t)(-1 - s);
            n++;
        }
        for (uint32_t m = t.dyn_made; m; m &= m - 1u) {
            const int r = __builtin_ctz(m);
            if (n >= MAX_MANIFOLDS) { over = true; continue; }
            if (!(t.dyn_kept >> r & 1u)) continue;
            h->mf_b0[n] = (int8_t)h->order[r];
            h->mf_b1[n] = (int8_t)p;
            n++;
        }
        if (over) h->overflow[p] |= RSG_STATUS_CONTACT_OVERFLOW;
    }

    // Whether any planned manifold can hold a point: false if all are of meshes
    // with no leaf about the ball.  (Ball-only arenas.)
    RSG_FN bool ball_meets() {
        const float r = make_ball_phys(A.ball.radius_uu, A.ball.mass).radius + 0.08f;
        const V3 lo = A.ball.b.pos - v3(r, r, r), hi = A.ball.b.pos + v3(r, r, r);
        for (int m = 0; m < h->n_mf; m++) {
            const int s = -1 - h->mf_b1[m];
            uint32_t at, end;
            if (!static_is_mesh(*geo, s) || leaf_list(geo->meshes[s].box_grid, lo, hi, at, end) != 0) return true;
        }
        return false;
    }

    // -----------------------------------------------------------------------
    // Narrowphase

    // The point to replace when all four are taken (sort_cached_points).
    RSG_FN static int replace_point(const TeamManifold& m, V3 n, float dist) {
        int max_pen = -1;
        float max_pen_d = dist;
        for (int i = 0; i < 4; i++)
            if (m.p[i].dist < max_pen_d) { max_pen = i; max_pen_d = m.p[i].dist; }
        const V3 p0 = m.p[0].la, p1 = m.p[1].la, p2 = m.p[2].la, p3 = m.p[3].la;
        const float r0 = max_pen != 0 ? fabsf(len2(cross(n - p1, p3 - p2))) : 0.f;
        const float r1 = max_pen != 1 ? fabsf(len2(cross(n - p0, p3 - p2))) : 0.f;
        const float r2 = max_pen != 2 ? fabsf(len2(cross(n - p0, p3 - p1))) : 0.f;
        const float r3 = max_pen != 3 ? fabsf(len2(cross(n - p0, p2 - p1))) : 0.f;
        int best = 0;
        float bv = r0;
        if (r1 > bv) { bv = r1; best = 1; }
        if (r2 > bv) { bv = r2; best = 2; }
        if (r3 > bv) { bv = r3; best = 3; }
        return best;
    }

    // A contact callback's effect on the arena: recorded, or applied at once
    // when the pair runs again in order.  Only two cars' pair can have more than
    // the record holds, and only it may run again: pair() finds all its
    // contacts, while those of a mesh and of the ball and a car come from the
    // rounds of search.  (These have one effect a pair at most: a car on the
    // world keeps its last, a car meets the ball in one point, a plane the ball
    // in one, and the ball's on a mesh are applied as they come.)
    static_assert(PAIR_EFFECTS >= 1, "one effect of any pair fits its record");
    RSG_FN void effect(TeamManifold& m, int mi, int& n_eff, bool direct, int kind, int a, int b, V3 v0, V3 v1) {
        const int code = kind | (a << 8) | (b << 16);
        // (the ball's against meshes come first in the pair order and are found in order)
        if (direct || (kind == EFF_BALL_WORLD && mesh_of(mi))) { team_apply_effect(A, code, v0, v1); return; }
        if (kind == EFF_CAR_WORLD && n_eff > 0) { m.eff_v = v0; return; }  // the flag is set either way, the last normal stays
        if (n_eff >= PAIR_EFFECTS) { m.redo = kind == EFF_CAR_CAR; return; }
        if (n_eff == 0 && kind != EFF_CAR_CAR) {
            m.eff_code = code;
            m.eff_v = v0;
        } else {
            Effect& e = g->log.eff[mi].e[n_eff];
            e.code = code;
            e.v0 = v0;
            e.v1 = v1;
        }
        n_eff++;
    }

    RSG_FN const MeshView* mesh_of(int mi) {
        const int b1 = h->mf_b1[mi], s = -1 - b1;
        return b1 < 0 && static_is_mesh(*geo, s) ? &geo->meshes[s] : nullptr;
    }
    // The first mesh manifold from mi on, or -1.
    RSG_FN int next_mesh(int mi) {
        for (; mi < h->n_mf; mi++)
            if (mesh_of(mi)) return mi;
        return -1;
    }
    RSG_FN TeamPair pair_of(int mi) {
        TeamPair q;
        q.b0 = h->mf_b0[mi];
        const int b1 = h->mf_b1[mi];
        q.thr = rs_min(w.threshold_of(q.b0), w.threshold_of(b1));
        q.respond = w.has_response(q.b0) && w.has_response(b1);
        q.x0 = q.cx = w.xf_of(q.b0);
        q.ball_r = make_ball_phys(A.ball.radius_uu, A.ball.mass).radius;
        q.he = v3zero();
        if (q.b0 > 0) {
            const CarPhys& cp = *A.cars[q.b0 - 1].phys;
            q.cx = w.car_child_xf(q.b0);
            q.he = cp.box_implicit + v3(cp.box_margin, cp.box_margin, cp.box_margin);
            const M3 ab = abs_m3(q.cx.R);
            const V3 e = v3(dot(ab.r[0], q.he), dot(ab.r[1], q.he), dot(ab.r[2], q.he));
            q.amin = q.cx.t - e;
            q.amax = q.cx.t + e;
        } else {
            const float r = q.ball_r + 0.08f;
            q.amin = q.x0.t - v3(r, r, r);
            q.amax = q.x0.t + v3(r, r, r);
        }
        return q;
    }
    // The manifold, empty.
    RSG_FN void open(int mi, const TeamPair& q) {
        const int b0 = q.b0, b1 = h->mf_b1[mi];
        TeamManifold& m = manifold(mi);
        float fa, ra, fb, rb;
        w.body_material(b0, fa, ra);
        w.body_material(b1, fb, rb);
        // combined friction / restitution (btManifoldResult.cpp:56-77), then
        // the contact callback's own
        float fr = b1 < 0 ? (fa < fb ? fa : fb) : fa * fb;
        float re = b1 < 0 ? (ra > rb ? ra : rb) : ra * rb;
        if (q.respond && b0 > 0) {
            if (b1 < 0) { fr = A.mut.car_world_friction; re = A.mut.car_world_restitution; }
            else if (b1 == 0) { fr = CARBALL_COLLISION_FRICTION; re = CARBALL_COLLISION_RESTITUTION; }
            else { fr = CARCAR_COLLISION_FRICTION; re = CARCAR_COLLISION_RESTITUTION; }
        }
        m.threshold = q.thr;
        m.friction = fr;
        m.restitution = re;
        m.special = q.respond && b0 == 0 && b1 < 0;
        m.redo = 0;
        m.n = 0;
        m.n_effects = 0;
    }
    // btManifoldResult::addContactPoint and the contact-added callback: body 1's
    // point pb, the normal on it and the distance; `tri` of a mesh's contact.
    RSG_FN void add_point(int mi, const TeamPair& q, V3 n, V3 pb, float dist, bool direct, const MeshView* mesh, int tri) {
        TeamManifold& m = manifold(mi);
        const int b0 = q.b0, b1 = h->mf_b1[mi];
        CPoint p;
        p.pos_a = pb + n * dist;
        p.pos_b = pb;
        p.local_a = xf_inv_apply(q.x0, p.pos_a);
        p.local_b = xf_inv_apply(w.xf_of(b1), pb);
        p.normal = n;
        p.dist = dist;
        int n_pts = m.n, n_eff = m.n_effects;
        const int idx = n_pts == MAX_POINTS_PER_MANIFOLD ? replace_point(m, p.local_a, dist) : n_pts++;
        if (q.respond) {
            if (b1 < 0) {
                if (b0 > 0) effect(m, mi, n_eff, direct, EFF_CAR_WORLD, b0 - 1, 0, p.normal, v3zero());
                else if (A.mode == RSG_MODE_HEATSEEKER) effect(m, mi, n_eff, direct, EFF_BALL_WORLD, 0, 0, p.normal, v3zero());
            } else if (b1 == 0) {
                effect(m, mi, n_eff, direct, EFF_CAR_BALL, b0 - 1, 0, p.local_b, v3zero());
            } else {
                effect(m, mi, n_eff, direct, EFF_CAR_CAR, b0 - 1, b1 - 1, p.local_a, p.local_b);
            }
            if (mesh) adjust_internal_edge(p, *mesh, tri);
        }
        TeamPoint& o = m.p[idx];
        o.la = p.local_a;
        o.lb = p.local_b;
        o.n = p.normal;
        o.dist = p.dist;
        m.n = (uint8_t)n_pts;
        m.n_effects = (uint8_t)n_eff;
    }
    // Manifold mi opened, with the contacts that need no search: a plane's, at
    // most one, or two cars' boxes', up to four.  (A mesh's and the ball's
    // against a car come in the rounds of contact().)
    RSG_FN void pair(int mi, bool direct) {
        const int b0 = h->mf_b0[mi], b1 = h->mf_b1[mi];
        const TeamPair q = pair_of(mi);
        open(mi, q);
        if (b1 == 0 || mesh_of(mi)) return;
        BoxBoxContacts bc;
        bc.n = 1;
        if (b1 > 0) {
            // copies for the call out of line: what it takes by reference
            // lives in memory
            const CarPhys& p1 = *A.cars[b1 - 1].phys;
            const Xf xa = q.cx, xb = w.car_child_xf(b1);
            const V3 half = q.he;
            BoxBoxContacts out;
            box_box(xa, half, xb, p1.box_implicit + v3(p1.box_margin, p1.box_margin, p1.box_margin), out);
            bc = out;
        }
        RSG_UNROLL_1
        for (int item = 0; item < bc.n; item++) {
            V3 n = bc.normal, pb = pick(item, bc.point[0], bc.point[1], bc.point[2], bc.point[3]);
            float dist = pick(item, bc.depth[0], bc.depth[1], bc.depth[2], bc.depth[3]);
            if (b1 < 0 && !plane_contact(b0, -1 - b1, q.cx, q.he, q.ball_r, q.thr, n, pb, dist)) continue;
            if (dist > q.thr) continue;
            add_point(mi, q, n, pb, dist, direct, nullptr, -1);
        }
    }

    // The rounds in which a team's lanes search contacts.  The first: the lane-th
    // manifold of a car and the ball, one a lane.  Then a mesh manifold after
    // the other, its triangles over the lanes.
    struct Search {
        int mi;        // the mesh manifold under way; before the first, -1
        bool more;     // rounds left
        TeamPair q;    // its pair (in the first round the lane's own)
        MeshBoxIter it;
    };
    // This lane's part of the next round: its manifold, or -1, and triangle
    // (-1: the ball).
    RSG_FN int next_search(Search& s, bool first, int& tri) {
        tri = -1;
        if (first) {
            s.mi = -1;
            s.it.mode = 0;
            int k = lane;
            int mine = -1;
            for (int m = 0; m < h->n_mf; m++)
                if (h->mf_b1[m] == 0 && k-- == 0) mine = m;
            s.more = next_mesh(0) >= 0;
            if (mine >= 0) s.q = pair_of(mine);
            return mine;
        }
        if (s.it.mode == 0) {
            s.mi = next_mesh(s.mi + 1);
            s.q = pair_of(s.mi);
            s.it.start(mesh_of(s.mi), s.q.amin, s.q.amax);
        }
        tri = s.it.next(lane, lanes);
        s.more = s.it.mode != 0 || next_mesh(s.mi + 1) >= 0;
        return tri >= 0 ? s.mi : -1;
    }
    // The lane's contact of the round: the closest points of body 0 (a car's
    // box, the ball's sphere) and its triangle or the ball.  1: there is one, 0:
    // none, -1: that takes the penetration pass, and there is no work space.
    RSG_FN int contact(const TeamPair& q, int mi, int tri, const EpaWork* first, const EpaWork* second, V3& n, V3& pb,
                       float& dist) {
        CShape other = shape_sphere(q.ball_r);
        Xf x1 = xf_ident();
        if (tri >= 0) {
            V3 v[3];
            mesh_triangle(*mesh_of(mi), tri, v);
            if (!triangle_aabb_overlap(v, q.amin, q.amax)) return 0;
            // early out on the triangle's plane, from both sides
            // (btConvexConcaveCollisionAlgorithm.cpp:86-125)
            const V3 tn = normalized(cross(v[1] - v[0], v[2] - v[0]));
            const M3 inv = inverse(q.cx.R);
            RSG_UNROLL_1
            for (int side = 0; side < 2; side++) {
                const V3 sn = side ? tn * -1.f : tn;
                const V3 d = inv * sn;
                V3 lp;
                if (q.b0 > 0) lp = v3(fsel(d.x, q.he.x, -q.he.x), fsel(d.y, q.he.y, -q.he.y), fsel(d.z, q.he.z, -q.he.z));
                else lp = (len2(d) < FLT_EPS * FLT_EPS) ? normalized(v3(-1, -1, -1)) * q.ball_r : q.ball_r * normalized(d);
                const V3 wp = xf_apply(q.cx, lp);
                const float gap = dot(sn, v[0]) - dot(sn, wp);
                if (gap > q.thr) return 0;
            }
            if (q.b0 == 0)
                return World::sphere_triangle_contact(q.x0.t, q.ball_r, q.thr, v, n, pb, dist) && !(dist > q.thr) ? 1 : 0;
            other = shape_triangle(v);
        } else {
            x1 = w.xf_of(0);
        }
        const CarPhys& cp = *A.cars[q.b0 - 1].phys;
        const CShape box = shape_box(cp.box_implicit, cp.box_margin);
        float md = box.margin + other.margin + q.thr;
        md *= md;
        const int r = gjk_closest(box, other, q.cx, x1, md, n, pb, dist, first, second);
        return r > 0 && dist > q.thr ? 0 : r;
    }

    // btPersistentManifold::refreshContactPoints (manifold_refresh).
    RSG_FN void refresh(int mi) {
        TeamManifold& m = manifold(mi);
        const float thr = m.threshold;
        const Xf x0 = w.xf_of(h->mf_b0[mi]), x1 = w.xf_of(h->mf_b1[mi]);
        int n_pts = m.n;
        RSG_UNROLL_1
        for (int i = n_pts - 1; i >= 0; i--) {
            const TeamPoint p = m.p[i];
            const V3 pa = xf_apply(x0, p.la), pb = xf_apply(x1, p.lb);
            const float d = dot(pa - pb, p.n);
            bool gone = !(d <= thr);
            if (!gone) {
                const V3 diff = pb - (pa - p.n * d);
                gone = dot(diff, diff) > thr * thr;
            }
            if (!gone) { m.p[i].dist = d; continue; }
            n_pts--;
            if (i != n_pts) m.p[i] = m.p[n_pts];
        }
        m.n = (uint8_t)n_pts;
    }
    RSG_FN void refresh_all() {
        RSG_UNROLL_1
        for (int mi = lane; mi < h->n_mf; mi += lanes) refresh(mi);
    }

    // btConvexPlaneCollisionAlgorithm::processCollision for the ball or a
    // car's box against static plane s.
    RSG_FN bool plane_contact(int b0, int s, const Xf& cx, V3 he, float ball_r, float thr, V3& n, V3& pb, float& dist) {
        const PlaneDef& pd = static_plane(*geo, s);
        const Xf px = xf_from(pd.origin, m3_identity());
        const Xf plane_in_convex = xf_mul(xf_inverse(cx), px);
        const Xf convex_in_plane = xf_mul(xf_inverse(px), cx);
        const V3 dir = plane_in_convex.R * -pd.n;
        V3 vtx;
        if (b0 > 0) vtx = v3(dir.x >= 0 ? he.x : -he.x, dir.y >= 0 ? he.y : -he.y, dir.z >= 0 ? he.z : -he.z);
        else if (len2(dir) < FLT_EPS * FLT_EPS) vtx = normalized(v3(-1, -1, -1)) * ball_r;
        else vtx = ball_r * normalized(dir);
        const V3 vin = xf_apply(convex_in_plane, vtx);
        dist = dot(pd.n, vin) - 0.f;
        if (!(dist < thr + 0.f)) return false;
        const V3 proj = vin - dist * pd.n;
        pb = xf_apply(px, proj);
        n = px.R * pd.n;
        return true;
    }

    // Pass 0: each lane its share of the manifolds; pass 1 (lane 0): the effects
    // in pair order, with the manifolds run again that had more than fit the
    // record.
    RSG_FN void narrow(int pass) {
        const int n = pass == 0 || lane == 0 ? h->n_mf : 0;
        RSG_UNROLL_1
        for (int mi = pass == 0 ? lane : 0; mi < n; mi += pass == 0 ? lanes : 1) {
            if (pass == 0 || manifold(mi).redo) {
                pair(mi, pass != 0);
                if (pass != 0) refresh(mi);
                continue;
            }
            const TeamManifold& m = manifold(mi);
            for (int j = 0; j < m.n_effects; j++) {
                const bool inl = j == 0 && (h->mf_b0[mi] <= 0 || h->mf_b1[mi] <= 0);
                int code;
                V3 v0, v1 = v3zero();
                if (inl) {
                    code = m.eff_code;
                    v0 = m.eff_v;
                } else {
                    const Effect& e = g->log.eff[mi].e[j];
                    code = e.code;
                    v0 = e.v0;
                    v1 = e.v1;
                }
                if ((code & 0xff) == EFF_CAR_WORLD) {
                    Car& c = A.cars[(code >> 8) & 0xff];
                    setflag(c.flags, RSG_CF_WORLD_CONTACT, true);
                    c.world_normal = v0;
                } else {
                    team_apply_effect(A, code, v0, v1);
                }
            }
        }
    }

    // -----------------------------------------------------------------------
    // Islands and solver

    // Nine small numbers in one register: 4 bits each, or 7.
    template <int BITS>
    struct Packed {
        uint64_t v;
        RSG_FN int get(int i) const { return (int)(v >> (BITS * i) & ((1u << BITS) - 1u)); }
        RSG_FN void set(int i, int x) {
            v = (v & ~((uint64_t)((1u << BITS) - 1u) << (BITS * i))) | (uint64_t)x << (BITS * i);
        }
    };
    static_assert(MAX_BODIES <= 9, "nine bodies' levels fit 63 bits");
    static_assert(MAX_ROWS <= 127 && MAX_MANIFOLDS <= 63, "row sources and levels are bytes");

    RSG_FN static int find(Packed<4>& id, int x) {
        while (x != id.get(x)) {
            id.set(x, id.get(id.get(x)));
            x = id.get(x);
        }
        return x;
    }

    // Union-find over the response pairs (World::island_unions).
    RSG_FN Packed<4> unions() {
        const int nb = bodies();
        Packed<4> id{0};
        for (int i = 0; i < nb; i++) id.set(i, i);
        for (int p = 0; p < nb; p++)
            for (uint32_t m = body[p].dyn; m; m &= m - 1u) {
                const int q = h->order[__builtin_ctz(m)];
                if (!w.has_response(p) || !w.has_response(q)) continue;
                const int i = find(id, p), j = find(id, q);
                if (i != j) id.set(i, j);
            }
        return id;
    }

    // quicksort_by_key over h->im with keys h->sort.key.
    RSG_FN void sort_manifolds(int n) {
        uint8_t* idx = h->im;
        const uint8_t* key = h->sort.key;
        int sp = 0;
        h->sort.lo[0] = 0; h->sort.hi[0] = (uint8_t)(n - 1); sp = 1;
        RSG_UNROLL_1
        while (sp > 0) {
            sp--;
            const int l = h->sort.lo[sp], hh = h->sort.hi[sp];
            int i = l, j = hh;
            const int x = key[idx[(l + hh) / 2]];
            do {
                while (key[idx[i]] < x) i++;
                while (x < key[idx[j]]) j--;
                if (i <= j) {
                    const uint8_t t = idx[i]; idx[i] = idx[j]; idx[j] = t;
                    i++; j--;
                }
            } while (i <= j);
            if (i < hh) { h->sort.lo[sp] = (uint8_t)i; h->sort.hi[sp] = (uint8_t)hh; sp++; }
            if (l < j) { h->sort.lo[sp] = (uint8_t)l; h->sort.hi[sp] = (uint8_t)j; sp++; }
        }
    }

    // Lane 0: the islands wake a sleeping ball, order the manifolds and give
    // the contact rows.  A row's level is one more than the highest level
    // among the earlier rows that share a dynamic body with it: rows of one
    // level touch different bodies, so running them side by side, level by
    // level, is the reference's row by row order.
    RSG_FN void rows() {
        if (lane != 0) return;
        h->n_rows = h->n_levels = 0;
        h->sp_num = 0;
        const int nb = bodies(), n_mf = h->n_mf;
        uint32_t dyn = 0;
        for (int p = 0; p < nb; p++) dyn |= body[p].dyn;
        bool any_point = false;
        for (int m = 0; m < n_mf; m++) any_point |= manifold(m).n > 0;
        Packed<4> id{0x876543210ull};
        if (dyn && (any_point || !A.ball.b.active)) id = unions();
        if (!A.ball.b.active) {
            const int root = find(id, 0);
            bool wake = false;
            for (int i = 1; i < nb; i++) wake |= A.cars[i - 1].b.active && find(id, i) == root;
            if (wake) A.ball.b.active = true;  // integrated, but got no gravity
        }
        if (!any_point) return;
        int n_im = 0;
        for (int m = 0; m < n_mf; m++) {
            const int b0 = h->mf_b0[m], b1 = h->mf_b1[m];
            const bool sleep0 = b0 == 0 && !A.ball.b.active, sleep1 = b1 < 0 || (b1 == 0 && !A.ball.b.active);
            if (sleep0 && sleep1) continue;
            if (!(w.has_response(b0) && w.has_response(b1))) continue;
            h->sort.key[m] = (uint8_t)find(id, b0);
            h->im[n_im++] = (uint8_t)m;
        }
        if (n_im > 1) sort_manifolds(n_im);
        int n = 0, levels = 0;
        bool over = false;
        Packed<7> next{0};  // the level after each body's last row
        V3 sp_normal = v3zero();
        float sp_dist = 0.f;
        int sp_num = 0;
        RSG_UNROLL_1
        for (int q = 0; q < n_im; q++) {
            const int mi = h->im[q];
            const TeamManifold& m = manifold(mi);
            const int b0 = h->mf_b0[mi], b1 = h->mf_b1[mi];
            if (heavy(b0) && (b1 < 0 || heavy(b1))) continue;
            for (int j = 0; j < m.n; j++) {
                if (n >= MAX_ROWS) { over = true; break; }
                int lv = next.get(b0);
                if (b1 >= 0 && next.get(b1) > lv) lv = next.get(b1);
                h->row.src[n] = (uint8_t)(mi | j << 6);
                h->row.level[n] = (uint8_t)lv;
                n++;
                lv++;
                next.set(b0, lv);
                if (b1 >= 0) next.set(b1, lv);
                if (lv > levels) levels = lv;
                if (m.special) {
                    const Body& bb = A.ball.b;
                    sp_num++;
                    h->sp_friction = m.friction;
                    h->sp_restitution = m.restitution;
                    sp_normal += m.p[j].n;
                    sp_dist += len(xf_apply(xf_from(bb.pos, bb.rot), m.p[j].la) - bb.pos);
                }
            }
        }
        if (sp_num > 0) {
            h->sp_num = sp_num;
            h->sp_normal = sp_normal;
            h->sp_dist = sp_dist;
            if (n >= MAX_ROWS) {
                over = true;
            } else {
                const int lv = next.get(0);
                h->row.src[n] = ROW_SPECIAL;
                h->row.level[n] = (uint8_t)lv;
                n++;
                if (lv + 1 > levels) levels = lv + 1;
            }
        }
        h->n_rows = n;
        h->n_levels = levels;
        if (over) A.status |= RSG_STATUS_SOLVER_OVERFLOW;
    }
    // btSequentialImpulseConstraintSolver::convertContact's test for a body
    // that contacts do not move.
    RSG_FN bool heavy(int code) {
        const float im = w.body_ptr(code)->inv_mass;
        return fuzzy_zero(v3(im, im, im));
    }

    // Row r's set-up (convertContactInner, convert_special).
    RSG_FN void row_setup(int r, float dt, TeamRow& row) {
        const int src = h->row.src[r];
        int b0, b1;
        V3 normal, rel1, rel2;
        float dist, friction, restitution;
        if (src == ROW_SPECIAL) {
            b0 = 0;
            b1 = -1;
            dist = h->sp_dist / (float)h->sp_num;
            normal = h->sp_normal * (1.f / (float)h->sp_num);
            friction = h->sp_friction;
            restitution = h->sp_restitution;
            rel1 = normal * -dist;
            rel2 = v3zero();
        } else {
            const int mi = src & 63;
            const TeamManifold& m = manifold(mi);
            b0 = h->mf_b0[mi];
            b1 = h->mf_b1[mi];
            const TeamPoint p = m.p[src >> 6];
            const Xf x0 = w.xf_of(b0), x1 = w.xf_of(b1);
            normal = p.n;
            dist = p.dist;
            friction = m.friction;
            restitution = m.restitution;
            rel1 = xf_apply(x0, p.la) - x0.t;
            rel2 = xf_apply(x1, p.lb) - x1.t;
        }
        row.a = b0;
        row.b = b1;
        const Body* rb0 = w.body_ptr(b0);
        const Body* rb1 = b1 >= 0 ? w.body_ptr(b1) : nullptr;
        SBody sa, sb;
        init_solver_body(sa, rb0->inv_mass != 0.f ? rb0 : nullptr, rb0->inv_mass != 0.f ? b0 : -1, dt);
        const bool dyn1 = rb1 && rb1->inv_mass != 0.f;
        init_solver_body(sb, dyn1 ? rb1 : nullptr, dyn1 ? b1 : -1, dt);
        setup_contact_row(sa, sb, dt, row.c, rb0, rb1, normal, dist, friction, restitution, rel1, rel2);
        row.c.special = src != ROW_SPECIAL && b0 == 0 && b1 < 0;
        setup_friction_row(sa, sb, row.f, rb0, rb1, friction_direction(sa, sb, normal, rel1, rel2), friction, rel1, rel2);
    }

    RSG_FN RowSide side(int code, bool push) {
        RowSide r{false, v3zero(), v3zero(), v3zero()};
        if (code < 0) return r;
        const float im = w.body_ptr(code)->inv_mass;
        if (im == 0.f) return r;
        r.dynamic = true;
        r.inv_mass = v3(im, im, im);
        r.lin = push ? body[code].push : body[code].dv;
        r.ang = push ? body[code].turn : body[code].dw;
        return r;
    }
    RSG_FN void put_side(int code, bool push, const RowSide& r) {
        if (!r.dynamic) return;
        if (push) { body[code].push = r.lin; body[code].turn = r.ang; }
        else { body[code].dv = r.lin; body[code].dw = r.ang; }
    }
    // One visit of a row: 0 its split-impulse row, 1 its contact row, 2 its
    // friction row.  Returns the split row's residual, the others' change.
    RSG_FN float row_visit(TeamRow& row, int what) {
        if (what == 0 && !(row.c.rhs_pen != 0.f)) return 0.f;
        if (what == 1 && row.c.special) return 0.f;
        if (what == 2 && !(row.c.applied > 0.f)) return 0.f;
        RowSide a = side(row.a, what == 0), b = side(row.b, what == 0);
        float r = 0.f;
        if (what == 0) {
            r = row_split(row.c, a, b);
        } else if (what == 1) {
            r = row_lower(row.c, a, b);
        } else {
            row.f.lo = -(row.f.friction * row.c.applied);
            row.f.hi = row.f.friction * row.c.applied;
            r = row_generic(row.f, a, b);
        }
        put_side(row.a, what == 0, a);
        put_side(row.b, what == 0, b);
        return r;
    }

    // -----------------------------------------------------------------------
    // The bodies' end of tick

    RSG_FN void body_end(const TickParams& P) {
        if (lane >= bodies()) return;
        const float dt = P.dt;
        Body& b = *w.body_ptr(lane);
        TeamBody& t = body[lane];
        if (b.active && b.inv_mass != 0.f) {
            // writeBackBodies
            const V3 ext_f = b.force * b.inv_mass * dt;
            const V3 ext_t = mul_vm(b.torque, b.inv_iw) * dt;
            if (t.push.x != 0.f || t.push.y != 0 || t.push.z != 0 || t.turn.x != 0.f || t.turn.y != 0 || t.turn.z != 0) {
                V3 np; M3 nr;
                integrate_transform(b.pos, b.rot, t.push, t.turn * SOLVER_SPLIT_TURN_ERP, dt, b.no_rot, np, nr);
                b.pos = np;
                b.rot = nr;
            }
            b.vel = (b.vel + t.dv) + ext_f;
            b.ang = (b.ang + t.dw) + ext_t;
        }
        w.body_integrate(lane, dt);
        if (lane == 0) {
            ball_finish(A);
        } else {
            car_post_tick(A, P, lane - 1);
            t.pad_window = pad_window(A, A.cars[lane - 1]);
        }
    }
    // The boost-pad grid cells within a car's reach (BoostPadGrid.cpp:5-25).
    RSG_FN static uint16_t pad_window(const ArenaLocal& A, const Car& c) {
        int x0, x1, y0, y1;
        if (!car_pad_window(A, c, x0, x1, y0, y1)) return TEAM_NO_PADS;
        if (x1 < 0 || y1 < 0 || x0 > 15 || y0 > 15) return TEAM_NO_PADS;
        return (uint16_t)(x0 | (x1 > 15 ? 15 : x1) << 4 | y0 << 8 | (y1 > 15 ? 15 : y1) << 12);
    }

    RSG_FN void pads(const TickParams& P) {
        if (!geo || A.n_cars == 0) return;
        for (int p = lane; p < A.n_pads; p += lanes) {
            Pad& pad = A.pads[p];
            pad_pre_tick(pad, P.dt);
            const int px = pad.cell & 15, py = pad.cell >> 4;
            for (int oi = 0; oi < A.n_cars; oi++) {
                const int ci = A.order[oi];
                if (!A.custom_pads) {
                    const int wn = body[1 + ci].pad_window;
                    if (px < (wn & 15) || px > (wn >> 4 & 15) || py < (wn >> 8 & 15) || py > (wn >> 12)) continue;
                }
                pad_check_collide(A, pad, p, A.cars[ci], ci, *A.cars[ci].phys);
            }
            if (pad.cur_locked >= 0) h->any_locked = 1;
            else pad.prev_locked = 0;
        }
    }
    RSG_FN void end(const TickParams& P) {
        if (lane != 0) return;
        if (h->any_locked)
            for (int p = 0; p < A.n_pads; p++)
                if (A.pads[p].cur_locked >= 0) pad_post_tick(A, p);
        uint32_t over = 0;
        for (int i = 0; i < bodies(); i++) over |= h->overflow[i];
        A.status |= over;
        if (tick_finish(A, P)) team_kickoff(A, P.seed, P.arena_id);
    }
};

}  // namespace rsg
