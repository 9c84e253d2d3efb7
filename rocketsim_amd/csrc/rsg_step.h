// rsg_step.h -- one arena stepped `ticks` ticks by one lane: gather the
// arena from the struct-of-arrays state, run Arena::Step's body
// (src/Sim/Arena/Arena.cpp:689-756) `ticks` times on the working copy, scatter
// it back.
#pragma once

#include "rsg_tick.h"

namespace rsg {

// Waves per SIMD the step kernels are compiled for (register budget).  The
// plain and LDS kernels run fastest with the whole register file (1).  The
// cooperative kernel waits on memory and on its slowest lane half of the time
// and gains from a second wave per SIMD where there are waves to fill it
// (2v2 x 16384 arenas: 0.350 ms a tick at 2, 0.415 at 1; 32768 arenas of 1v1
// to 3v3: 0.587 and 0.940), and loses a little to its spills where there are
// not (2v2 x 4096: 0.192 and 0.183).
#ifndef RSG_STEP_WAVES_PER_EU
#define RSG_STEP_WAVES_PER_EU 1
#endif
#ifndef RSG_COOP_WAVES_PER_EU
#define RSG_COOP_WAVES_PER_EU 2
#endif

// Arena `a`'s block of the batch's global work space.
RSG_FN StepSpace* arena_space(const BatchDev& d, int a) {
    return &reinterpret_cast<ArenaSpace*>(d.space)[a].step;
}

RSG_FN void step_arena(const BatchDev& d, const ArenaGeom& geom, int a, int ticks, ArenaLocal& A, StepSpace* ws) {
    load_arena(d, a, A);
    TickParams P;
    P.mode = d.mode;
    P.dt = d.tick_time;
    P.seed = d.seed;
    P.arena_id = (uint32_t)a;
    P.synth_controls = d.synth_controls != 0;
    P.auto_reset = d.auto_reset != 0;
    const ArenaGeom* mp = mode_has_arena(d.mode) ? &geom : nullptr;
    for (int t = 0; t < ticks; t++) arena_tick(A, P, mp, ws);
    store_arena(d, a, A);
}

}  // namespace rsg
