// Host run of the team tick (rocketsim_amd/csrc/rsg_team.h), phase by phase
// and lane by lane, as the cooperative kernel's lanes run it; th_step of
// tick_host.cpp with the phases in place of arena_tick.
#include <memory>
#include <vector>
#define th_step th_step_serial
#include "tick_host.cpp"
#undef th_step
#include "../../rocketsim_amd/csrc/rsg_team.h"

namespace {
// The lanes run last to first in every phase (none depends on another's).
template <class F>
void each_lane(ArenaLocal& A, const ArenaGeom* geo, unsigned char* local, int max_cars, TeamGlobal* g, int lanes, F&& f) {
    for (int k = lanes - 1; k >= 0; k--) {
        Team t(A, geo, local, max_cars, g, k, lanes);
        f(t);
    }
}
}  // namespace

void team_tick(ArenaLocal& A, const TickParams& P, const ArenaGeom* geo, unsigned char* local, int max_cars,
               TeamGlobal* g, int lanes) {
    auto each = [&](auto&& f) { each_lane(A, geo, local, max_cars, g, lanes, f); };
    TeamHead* h = reinterpret_cast<TeamHead*>(local);
    each([&](Team& t) { t.begin(P); });
    Team t0(A, geo, local, max_cars, g, 0, lanes);
    const bool respawn = t0.any_respawn();
    if (!respawn) each([&](Team& t) { t.rays(-1); });
    const bool together = !respawn && t0.independent();
    for (int pass = 0; pass < t0.car_passes(together); pass++) {
        each([&](Team& t) { t.car_begin(P, together, pass); });
        if (respawn) each([&](Team& t) { t.rays(pass); });
        each([&](Team& t) { t.wheels(P, together, pass); });
        each([&](Team& t) { t.car(P, together, pass); });
    }
    each([&](Team& t) { t.body_begin(P); });
    each([&](Team& t) { t.ranks(); });
    each([&](Team& t) { t.pairs(); });
    each([&](Team& t) { t.trim(); });
    each([&](Team& t) { t.drop_pairs(); });
    each([&](Team& t) { t.plan(); });
    each([&](Team& t) { t.narrow(0); });
    EpaSmall small;
    struct Found { int mi, tri, found; V3 n, pb; float dist; };
    std::vector<Team::Search> search((size_t)lanes);
    std::vector<Found> f((size_t)lanes);
    bool first = true, more = true;
    while (more) {
        more = false;
        each([&](Team& t) {
            Found& o = f[(size_t)t.lane];
            o.mi = t.next_search(search[(size_t)t.lane], first, o.tri);
            more |= search[(size_t)t.lane].more;
            o.found = 0;
            const EpaWork w0 = epa_work(small), w1 = epa_work(t.g->epa);
            for (int turn = 0; turn < 2 && o.mi >= 0 && (turn == 0 || o.found < 0); turn++)
                o.found = t.contact(search[(size_t)t.lane].q, o.mi, o.tri, turn ? &w0 : nullptr, &w1, o.n, o.pb, o.dist);
        });
        first = false;
        for (int k = 0; k < lanes; k++) {
            if (f[(size_t)k].found <= 0) continue;
            Team t(A, geo, local, max_cars, g, k, lanes);
            const Found& o = f[(size_t)k];
            t.add_point(o.mi, search[(size_t)k].q, o.n, o.pb, o.dist, false, o.tri >= 0 ? t.mesh_of(o.mi) : nullptr, o.tri);
        }
    }
    each([&](Team& t) { t.refresh_all(); });
    each([&](Team& t) { t.narrow(1); });
    each([&](Team& t) { t.rows(); });
    const int n = h->n_rows;
    std::vector<TeamRow> rows((size_t)n);
    for (int r = 0; r < n; r++) t0.row_setup(r, P.dt, rows[(size_t)r]);
    auto visit = [&](int what) {
        bool moved = false;
        for (int lv = 0; lv < h->n_levels; lv++)
            for (int r = n - 1; r >= 0; r--)
                if (h->row.level[r] == lv) {
                    const float q = t0.row_visit(rows[(size_t)r], what);
                    moved |= what == 0 ? !(q * q <= 0.f) : q != 0.f;
                }
        return moved;
    };
    for (int it = 0; it < SOLVER_ITERATIONS; it++)
        if (!visit(0)) break;
    for (int it = 0; it < SOLVER_ITERATIONS; it++) {
        const bool contacts = visit(1), friction = visit(2);
        if (!contacts && !friction) break;
    }
    each([&](Team& t) { t.body_end(P); });
    each([&](Team& t) { t.pads(P); });
    each([&](Team& t) { t.end(P); });
}

extern "C" void th_step(void* p, int ticks) {
    HostBatch& h = *(HostBatch*)p;
    const ArenaGeom mv = h.geo.geom();
    const ArenaGeom* mp = mode_has_arena(h.dev.mode) ? &mv : nullptr;
    auto A = std::make_unique<ArenaLocal>();
    auto g = std::make_unique<ArenaSpace>();
    const int max_cars = h.dev.max_cars, lanes = 4 * max_cars < 12 ? 12 : 4 * max_cars;
    std::vector<uint64_t> local(team_local_bytes(max_cars) / 8 + 1);
    for (int a = 0; a < h.dev.n; a++) {
        load_arena(h.dev, a, *A);
        TickParams P;
        P.mode = h.dev.mode;
        P.dt = h.dev.tick_time;
        P.seed = h.dev.seed;
        P.arena_id = (uint32_t)a;
        P.synth_controls = h.dev.synth_controls != 0;
        P.auto_reset = h.dev.auto_reset != 0;
        for (int t = 0; t < ticks; t++)
            team_tick(*A, P, mp, (unsigned char*)local.data(), max_cars, reinterpret_cast<TeamGlobal*>(g.get()), lanes);
        store_arena(h.dev, a, *A);
    }
}
