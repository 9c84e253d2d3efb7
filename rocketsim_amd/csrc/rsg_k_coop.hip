// rsg_k_coop.hip -- the cooperative step kernel: a team of lanes (4 per car
// slot) per arena runs the phases of rsg_team.h, the arena's working copy and
// the tick's tables in LDS.
#include <hip/hip_runtime.h>

#include "rsg_kernels.h"
#include "rsg_step.h"
#include "rsg_team_wave.h"

using namespace rsg;

// `lanes` lanes per arena, at most 64 per workgroup: a workgroup is one wave,
// so its barriers only order the LDS accesses.
__global__ void __launch_bounds__(64) __attribute__((amdgpu_waves_per_eu(RSG_COOP_WAVES_PER_EU)))
rsg_step_arena_coop_kernel(BatchDev d, const ArenaGeom* geo, int ticks, int stride, int arena_bytes, int lanes) {
    extern __shared__ __align__(16) unsigned char rsg_lds[];
    const int slot = (int)threadIdx.x / lanes;
    const int k = (int)threadIdx.x - slot * lanes;
    const int a = (int)blockIdx.x * ((int)blockDim.x / lanes) + slot;
    const bool live = a < d.n;
    unsigned char* base = rsg_lds + (size_t)slot * (size_t)stride;
    ArenaLocal& A = *reinterpret_cast<ArenaLocal*>(base);
    TickParams P;
    P.mode = d.mode;
    P.dt = d.tick_time;
    P.seed = d.seed;
    P.arena_id = (uint32_t)a;
    P.synth_controls = d.synth_controls != 0;
    P.auto_reset = d.auto_reset != 0;
    const bool has_arena = geo != nullptr;
    TeamGlobal* g = reinterpret_cast<TeamGlobal*>(&reinterpret_cast<ArenaSpace*>(d.space)[live ? a : 0]);
    // The team, made anew for each phase from values the compiler cannot see
    // through: what a phase derives from them (addresses, geometry) then lives
    // for that phase alone.  Left to itself the compiler hoists all phases'
    // invariants out of the tick loop, and at 256 registers that costs 260
    // spilled registers and 400 reloads a tick.
    auto team = [&]() {
        unsigned off = (unsigned)slot * (unsigned)stride;
        int lane = k, team_lanes = lanes;
        const ArenaGeom* statics = geo;
        TeamGlobal* space = g;
        asm volatile("" : "+v"(off), "+v"(lane), "+s"(statics), "+s"(team_lanes), "+v"(space));
        unsigned char* at = rsg_lds + off;
        return Team(*reinterpret_cast<ArenaLocal*>(at), statics, at + arena_bytes, d.max_cars, space, lane, team_lanes);
    };
    // after the arenas' blocks: the wave's penetration work space
    EpaSmall* small = reinterpret_cast<EpaSmall*>(rsg_lds + (size_t)(blockDim.x / lanes) * (size_t)stride);
    const uint64_t team_mask = (lanes < 64 ? (1ull << lanes) - 1ull : ~0ull) << (slot * lanes);
    // pairs can pass the capacity only with many statics
    const int most_pairs = MAX_BODIES * (has_arena ? num_statics(*geo) : 0) + MAX_BODIES * (MAX_BODIES - 1) / 2;

    if (live && k == 0) load_arena_scalars(d, a, A);
    __syncthreads();
    if (live && k < A.n_cars) load_arena_car(d, a, A, k);
    if (live && has_arena)
        for (int p = k; p < PAD_NUM; p += lanes) load_arena_pad(d, a, A, p);
    __syncthreads();
    RSG_UNROLL_1
    for (int tick = 0; tick < ticks; tick++) {
        if (live) team().begin(P);
        __syncthreads();
        const bool respawn = live && team().any_respawn();
        bool together = false;
        int passes = 0;
        // pass -1 casts every ray ahead of the cars' updates, unless a car
        // respawns; then each pass casts its car's
        RSG_UNROLL_1
        for (int pass = -1; pass < 0 || __any(pass < passes); pass++) {
            const bool on = pass < 0 ? live : pass < passes;
            if (on && pass >= 0) team().car_begin(P, together, pass);
            __syncthreads();
            if (on && respawn == (pass >= 0)) team().rays(pass);
            __syncthreads();
            if (pass < 0) {
                together = live && !respawn && team().independent();
                passes = live ? team().car_passes(together) : 0;
                continue;
            }
            if (on) team().wheels(P, together, pass);
            __syncthreads();
            if (on) team().car(P, together, pass);
            __syncthreads();
        }
        if (live) team().body_begin(P);
        __syncthreads();
        if (live) team().ranks();
        __syncthreads();
        if (live) team().pairs();
        __syncthreads();
        if (most_pairs > MAX_PAIRS) {
            if (live) team().trim();
            __syncthreads();
            if (live) team().drop_pairs();
            __syncthreads();
        }
        if (live) team().plan();
        __syncthreads();
        team_narrow(team, live, small, team_mask);
        if (live) team().rows();
        __syncthreads();
        {
            Team t = team();
            team_solve(t, live, P.dt, team_mask);
        }
        __syncthreads();
        if (live) team().body_end(P);
        __syncthreads();
        if (live) team().pads(P);
        __syncthreads();
        if (live) team().end(P);
        __syncthreads();
    }
    if (live && k == 0) store_arena_scalars(d, a, A);
    if (live && k < A.n_cars) store_arena_car(d, a, A, k);
    if (live && has_arena)
        for (int p = k; p < PAD_NUM; p += lanes) store_arena_pad(d, a, A, p);
}

namespace rsg {

hipError_t launch_step_coop(const BatchDev& d, const ArenaGeom* geo, int ticks, int grid, int per_block, int stride,
                            int arena_bytes, int lanes, hipStream_t s) {
    const size_t lds = (size_t)per_block * (size_t)stride + sizeof(EpaSmall);
    hipLaunchKernelGGL(rsg_step_arena_coop_kernel, dim3(grid), dim3(per_block * lanes), lds, s, d, geo, ticks,
                       stride, arena_bytes, lanes);
    return hipGetLastError();
}

}  // namespace rsg
