// rsg_k_pred.hip -- the ball-prediction kernel (BallPredTracker updates,
// rsg_ball_pred.h).
#include <hip/hip_runtime.h>

#include "rsg_kernels.h"
#include "rsg_step.h"
#include "rsg_team_wave.h"

using namespace rsg;

namespace {
// Word w of the ball's record (pred_put), by the ball's place in memory.
static_assert(offsetof(Body, rot) == offsetof(Body, pos) + 12 && offsetof(Body, vel) == offsetof(Body, pos) + 48 &&
              offsetof(Body, ang) == offsetof(Body, pos) + 60, "position, basis and velocities lie in a row");
static_assert(RSG_PRED_WORDS == 23, "a record's words");
__device__ __forceinline__ uint32_t pred_word(const Ball& ball, int w) {
    const float* f = &ball.b.pos.x;
    if (w < 18) {
        const int row = (w - 3) % 3, col = (w - 3) / 3;
        const float x = f[w >= 3 && w < 12 ? 3 + row * 3 + col : w];
        return fw(w < 3 || (w >= 12 && w < 15) ? x * BT_TO_UU : x);
    }
    if (w == 18) return (uint32_t)ball.ticks_since_set;
    if (w == 19) return (uint32_t)(ball.ticks_since_set >> 32);
    return fw(w == 20 ? ball.hs_dir : (w == 21 ? ball.hs_speed : ball.hs_time));
}
}  // namespace

// One update of every tracker: a team of `lanes` lanes each, `per_wave` teams
// a workgroup (one wave), which run the ball-only tick in the phases of
// rsg_team.h.  Tracker i's prediction arena (arena i of `pa`) is held in LDS,
// `stride` bytes a tracker, the team's block from `arena_bytes` on.
//
// What bounds it: latency, as every tick waits for the one before.  A ball
// that meets nothing this tick (its planned manifolds are of meshes with no
// leaf about it) goes from the broadphase straight to the integration.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RSG_COOP_WAVES_PER_EU)))
rsg_ball_pred_kernel(BatchDev pa, const ArenaGeom* geo, PredDev p, int kind, BatchDev src, int stride, int arena_bytes,
                     int per_wave, int lanes) {
    extern __shared__ __align__(16) unsigned char rsg_lds[];
    const int slot = (int)threadIdx.x / lanes;
    const int k = (int)threadIdx.x - slot * lanes;
    const int i = (int)blockIdx.x * per_wave + slot;
    const bool live = i < pa.n;
    ArenaLocal& A = *reinterpret_cast<ArenaLocal*>(rsg_lds + (size_t)slot * (size_t)stride);
    EpaSmall* small = reinterpret_cast<EpaSmall*>(rsg_lds + (size_t)per_wave * (size_t)stride);
    TeamGlobal* g = reinterpret_cast<TeamGlobal*>(&reinterpret_cast<ArenaSpace*>(pa.space)[live ? i : 0]);
    const TickParams P = pred_tick_params(pa, i);
    const uint64_t team_mask = (lanes < 64 ? (1ull << lanes) - 1ull : ~0ull) << (slot * lanes);
    // the team, made anew for each phase (see rsg_k_coop.hip)
    auto team = [&]() {
        unsigned off = (unsigned)slot * (unsigned)stride;
        int lane = k, team_lanes = lanes;
        const ArenaGeom* statics = geo;
        TeamGlobal* space = g;
        asm volatile("" : "+v"(off), "+v"(lane), "+s"(statics), "+s"(team_lanes), "+v"(space));
        unsigned char* at = rsg_lds + off;
        return Team(*reinterpret_cast<ArenaLocal*>(at), statics, at + arena_bytes, 1, space, lane, team_lanes);
    };

    const size_t s = (size_t)pa.n;
    PredRun r{0, 0, false, false, 0};
    uint32_t cur[RSG_PRED_WORDS];
    if (live) r = pred_begin(p, kind, src, i, s, cur);
    __syncthreads();  // every lane has read the ring
    if (live && k == 0) {
        load_arena_scalars(pa, i, A);
        pred_start(p, r, i, s, cur, A.ball);
    }
    int t = !live || !(r.fresh || r.from_last) ? p.T : (r.fresh ? 1 : r.size);
    int row = live ? (r.head + t) % p.T : 0;
    __syncthreads();
    RSG_UNROLL_1
    while (__any(t < p.T)) {
        const bool on = t < p.T;
        bool meets = false;
        if (on && k == 0) {
            Team b = team();
            b.begin(P);
            b.body_begin(P);
            b.ranks();
            b.pairs();
            b.plan();
            b.h->n_rows = b.h->n_levels = 0;
            meets = b.h->n_mf > 0 && b.ball_meets();
        }
        __syncthreads();
        const uint64_t meeting = __ballot(meets);
        if (meeting) {
            const bool in = (meeting & team_mask) != 0;
            team_narrow(team, in, small, team_mask);
            if (in) team().rows();
            __syncthreads();
            {
                Team b = team();
                team_solve(b, in, P.dt, team_mask);
            }
            __syncthreads();
        }
        if (on && k == 0) {
            Team b = team();
            b.body_end(P);
            b.h->any_locked = 0;
            b.end(P);
        }
        __syncthreads();
        if (on) {
            uint32_t* out = p.traj + i + (size_t)row * RSG_PRED_WORDS * s;
            for (int w = k; w < RSG_PRED_WORDS; w += lanes) out[w * s] = pred_word(A.ball, w);
            t++;
            row = row + 1 == p.T ? 0 : row + 1;
        }
        __syncthreads();
    }
    if (live && k == 0) {
        pred_end(p, kind, r, i);
        store_arena_scalars(pa, i, A);
    }
}

namespace rsg {

hipError_t launch_ball_pred(const BatchDev& pa, const ArenaGeom* geo, const PredDev& p, int kind, const BatchDev& src,
                            int stride, int arena_bytes, int per_wave, int lanes, int grid, hipStream_t s) {
    const size_t lds = (size_t)per_wave * (size_t)stride + sizeof(EpaSmall);
    hipLaunchKernelGGL(rsg_ball_pred_kernel, dim3(grid), dim3(per_wave * lanes), lds, s, pa, geo, p, kind, src, stride,
                       arena_bytes, per_wave, lanes);
    return hipGetLastError();
}

}  // namespace rsg
