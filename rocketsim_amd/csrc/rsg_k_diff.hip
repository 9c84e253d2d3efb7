// rsg_k_diff.hip -- kernels of the differentiable rollouts: the airborne
// car (rsg_adjoint.h) and the aerial shot through the car-ball hit
// (rsg_shot.h), forward with checkpoints and backward.
#include <hip/hip_runtime.h>

#include "rsg_kernels.h"
#include "rsg_tick.h"
#include "rsg_adjoint.h"
#include "rsg_shot.h"

using namespace rsg;

// ---------------------------------------------------------------------------
// Airborne-car rollouts and their adjoint (rsg_adjoint.h).  One lane per car.
// Arrays come by word (state [13][n]: position uu, quaternion x y z w, velocity
// uu/s, angular velocity rad/s; controls [ticks][4][n]: pitch, yaw, roll, boost;
// target [7][n]: quaternion, position uu) or, with ROWS, by car (state [n][13],
// controls [ticks][n][4], target [n][7]); checkpoints [ceil(ticks / K)][13][n]
// in Bullet units either way.
//
// What bounds them: the chain of ticks, 1 us forward and 2 us for the adjoint,
// at one wave per SIMD (65536 cars: 309 and 756 VALU instructions a tick, whose
// issue takes 45 and 72 % of the wave's cycles; it waits 37 and 14 %); and
// memory where whole arrays are passed over again.
// By car, controls are read and their gradient written as 16 bytes a lane
// where the caller has them, with no transposed copies (65536 cars x 120 ticks:
// 130 us).  With K = 1 the adjoint reads each tick's state, a tick ahead of its
// use, instead of computing the segment again into private memory (303 us against
// 390; 257 cars x 45 ticks 88 against 134).

// Word w of car i.
template <bool ROWS, int WORDS>
RSG_FN size_t air_at(int w, int n, int i) {
    return ROWS ? (size_t)i * WORDS + w : (size_t)w * n + i;
}

template <bool ROWS>
RSG_FN AirState air_load(const float* a, int n, int i, bool uu) {
    float k = uu ? UU_TO_BT : 1.f;
    auto x = [&](int w) { return a[air_at<ROWS, AIR_STATE_WORDS>(w, n, i)]; };
    AirState s;
    s.p = v3(x(0), x(1), x(2)) * k;
    s.q = q4(x(3), x(4), x(5), x(6));
    s.v = v3(x(7), x(8), x(9)) * k;
    s.w = v3(x(10), x(11), x(12));
    return s;
}

template <bool ROWS>
RSG_FN void air_store(float* a, int n, int i, const AirState& s, float kpv) {
    auto put = [&](int w, float x) { a[air_at<ROWS, AIR_STATE_WORDS>(w, n, i)] = x; };
    put(0, s.p.x * kpv); put(1, s.p.y * kpv); put(2, s.p.z * kpv);
    put(3, s.q.x); put(4, s.q.y); put(5, s.q.z); put(6, s.q.w);
    put(7, s.v.x * kpv); put(8, s.v.y * kpv); put(9, s.v.z * kpv);
    put(10, s.w.x); put(11, s.w.y); put(12, s.w.z);
}

template <bool ROWS>
RSG_FN AirCtrl air_ctrl(const float* c, int n, int i, int t) {
    const float* b = c + (size_t)t * 4 * n;
    auto x = [&](int w) { return b[air_at<ROWS, 4>(w, n, i)]; };
    AirCtrl k;
    k.pitch = x(0); k.yaw = x(1); k.roll = x(2); k.boost = x(3);
    return k;
}
template <bool ROWS>
RSG_FN void air_put_ctrl(float* c, int n, int i, int t, const AirCtrl& k) {
    float* b = c + (size_t)t * 4 * n;
    b[air_at<ROWS, 4>(0, n, i)] = k.pitch; b[air_at<ROWS, 4>(1, n, i)] = k.yaw;
    b[air_at<ROWS, 4>(2, n, i)] = k.roll; b[air_at<ROWS, 4>(3, n, i)] = k.boost;
}

template <bool ROWS>
RSG_FN void air_target(const float* a, int n, int i, Q4& q, V3& p) {
    auto x = [&](int w) { return a[air_at<ROWS, 7>(w, n, i)]; };
    q = q4(x(0), x(1), x(2), x(3));
    p = v3(x(4), x(5), x(6)) * UU_TO_BT;
}

// Ticks whose loads are issued together, a group ahead of their use: loads wait
// for the stores issued before them, which are then a whole group old (65536
// cars x 120 ticks, forward with every state kept: 156 us against 213 at one
// tick ahead, backward 303 against 309).
constexpr int AIR_AHEAD = 4;

// `kept` and `kept_target` (by car, or null): copies of the controls and the
// target for the backward pass.
template <bool ROWS>
__global__ void __launch_bounds__(64) rsg_air_forward_kernel(int n, int ticks, int K, float dt, const float* s0,
                                                             const float* ctrl, const float* target, float* s_out,
                                                             float* loss, float* ckpt, float* kept,
                                                             float* kept_target) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    AirState s = air_load<ROWS>(s0, n, i, true);
    auto ctrl_at = [&](int t) { return air_ctrl<ROWS>(ctrl, n, i, t < ticks ? t : ticks - 1); };
    AirCtrl c[AIR_AHEAD], next[AIR_AHEAD];
    for (int k = 0; k < AIR_AHEAD; k++) c[k] = ctrl_at(k);
    int in_seg = 0;
    RSG_UNROLL_1
    for (int t0 = 0; t0 < ticks; t0 += AIR_AHEAD) {
        for (int k = 0; k < AIR_AHEAD; k++) next[k] = ctrl_at(t0 + AIR_AHEAD + k);
        RSG_UNROLL
        for (int k = 0; k < AIR_AHEAD; k++) {
            if (t0 + k >= ticks) break;
            if (ckpt && in_seg == 0) {
                air_store<false>(ckpt, n, i, s, 1.f);
                ckpt += (size_t)AIR_STATE_WORDS * n;
            }
            in_seg = in_seg + 1 == K ? 0 : in_seg + 1;
            if (kept) air_put_ctrl<ROWS>(kept, n, i, t0 + k, c[k]);
            air_step(s, c[k], dt);
        }
        for (int k = 0; k < AIR_AHEAD; k++) c[k] = next[k];
    }
    if (s_out) air_store<ROWS>(s_out, n, i, s, BT_TO_UU);
    if (kept_target)
        for (int w = 0; w < 7; w++) kept_target[air_at<ROWS, 7>(w, n, i)] = target[air_at<ROWS, 7>(w, n, i)];
    if (loss) {
        Q4 tq; V3 tp;
        air_target<ROWS>(target, n, i, tq, tp);
        loss[i] = air_loss(s, tq, tp);
    }
}

template <bool ROWS>
__global__ void __launch_bounds__(64) rsg_air_backward_kernel(int n, int ticks, int K, float dt, const float* ctrl,
                                                              const float* target, const float* ckpt,
                                                              const float* dloss, float* dctrl, float* ds0) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    const int nseg = (ticks + K - 1) / K;
    AirState st[AIR_MAX_K];
    // final state: recompute the last segment from its checkpoint
    AirState s = air_load<false>(ckpt + (size_t)(nseg - 1) * AIR_STATE_WORDS * n, n, i, false);
    for (int t = (nseg - 1) * K; t < ticks; t++) air_step(s, air_ctrl<ROWS>(ctrl, n, i, t), dt);
    Q4 tq; V3 tp;
    air_target<ROWS>(target, n, i, tq, tp);
    AirState g;
    air_loss_grad(s, tq, tp, dloss[i], g);
    for (int seg = nseg - 1; seg >= 0; seg--) {
        int t0 = seg * K, t1 = t0 + K < ticks ? t0 + K : ticks;
        AirState x = air_load<false>(ckpt + (size_t)seg * AIR_STATE_WORDS * n, n, i, false);
        for (int t = t0; t < t1; t++) {
            st[t - t0] = x;
            air_step(x, air_ctrl<ROWS>(ctrl, n, i, t), dt);
        }
        for (int t = t1 - 1; t >= t0; t--) {
            AirCtrl gc = {0.f, 0.f, 0.f, 0.f};
            air_step_adjoint(st[t - t0], air_ctrl<ROWS>(ctrl, n, i, t), dt, g, gc);
            air_put_ctrl<ROWS>(dctrl, n, i, t, gc);
        }
    }
    // initial-state gradient in interface units (uu for position and velocity)
    if (ds0) air_store<ROWS>(ds0, n, i, g, UU_TO_BT);
}

// The same with every tick's state at hand (K = 1).
template <bool ROWS>
__global__ void __launch_bounds__(64) rsg_air_backward_kept_kernel(int n, int ticks, float dt, const float* ctrl,
                                                                   const float* target, const float* ckpt,
                                                                   const float* dloss, float* dctrl, float* ds0) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    auto state = [&](int t) { return air_load<false>(ckpt + (size_t)t * AIR_STATE_WORDS * n, n, i, false); };
    auto ctrl_at = [&](int t) { return air_ctrl<ROWS>(ctrl, n, i, t); };
    AirState x[AIR_AHEAD], xn[AIR_AHEAD];
    AirCtrl c[AIR_AHEAD], cn[AIR_AHEAD];
    for (int k = 0; k < AIR_AHEAD; k++) {
        const int t = ticks - 1 - k < 0 ? 0 : ticks - 1 - k;
        x[k] = state(t);
        c[k] = ctrl_at(t);
    }
    AirState s = x[0];
    air_step(s, c[0], dt);
    Q4 tq; V3 tp;
    air_target<ROWS>(target, n, i, tq, tp);
    AirState g;
    air_loss_grad(s, tq, tp, dloss[i], g);
    RSG_UNROLL_1
    for (int t1 = ticks - 1; t1 >= 0; t1 -= AIR_AHEAD) {
        for (int k = 0; k < AIR_AHEAD; k++) {
            const int t = t1 - AIR_AHEAD - k < 0 ? 0 : t1 - AIR_AHEAD - k;
            xn[k] = state(t);
            cn[k] = ctrl_at(t);
        }
        RSG_UNROLL
        for (int k = 0; k < AIR_AHEAD; k++) {
            if (t1 - k < 0) break;
            AirCtrl gc = {0.f, 0.f, 0.f, 0.f};
            air_step_adjoint(x[k], c[k], dt, g, gc);
            air_put_ctrl<ROWS>(dctrl, n, i, t1 - k, gc);
        }
        for (int k = 0; k < AIR_AHEAD; k++) {
            x[k] = xn[k];
            c[k] = cn[k];
        }
    }
    if (ds0) air_store<ROWS>(ds0, n, i, g, UU_TO_BT);
}

// Differentiable aerial shot (rsg_shot.h): one lane per car-ball pair.
__global__ void __launch_bounds__(256) rsg_shot_forward_kernel(int n, int ticks, int K, float dt, const float* state0,
                                                               const float* ctrl, const float* target,
                                                               float* state_out, float* loss, float* ckpt,
                                                               uint32_t* flags) {
    int i = blockIdx.x * blockDim.x + threadIdx.x;
    if (i >= n) return;
    ShotConsts k = shot_consts(dt);
    ShotState<float> s;
    shot_load(state0, n, i, s);
    uint32_t fl = 0;
    V3 tg = v3(target[i], target[n + i], target[2 * n + i]);
    float l = shot_forward(s, ctrl, n, i, ticks, K, ckpt, tg, k, fl);
    if (state_out) shot_store(state_out, n, i, s);
    if (loss) loss[i] = l;
    if (flags) flags[i] = fl;
}

// Backward of the shot: one group of SHOT_GROUP lanes per pair, lane j < 26
// carrying the tangent along input j of every tick (22 state words, then
// pitch, yaw, roll, boost), so a pair's 26 passes per tick run side by side
// instead of one after another.  Every lane of a group recomputes the same
// segment from its checkpoint; lane 0 keeps the segment's states in LDS
// ([K][SHOT_LDS_WORDS] per group), and after each tick the group gathers the
// new state adjoint from lanes 0-21 with cross-lane shuffles.  A group spans
// half a wave, so no workgroup barrier is needed: a group whose pair is past
// n leaves at once.
constexpr int SHOT_GROUP = 32;
constexpr int SHOT_LDS_WORDS = 24;   // a checkpoint's 23 words, padded

__global__ void __launch_bounds__(256) rsg_shot_backward_kernel(int n, int ticks, int K, float dt, const float* ctrl,
                                                                const float* target, const float* ckpt,
                                                                const float* dloss, float* dctrl, float* ds0) {
    extern __shared__ float shot_seg[];
    const int lane = threadIdx.x & (SHOT_GROUP - 1);
    const int grp = threadIdx.x / SHOT_GROUP;
    const int i = blockIdx.x * (blockDim.x / SHOT_GROUP) + grp;
    if (i >= n) return;
    float* seg = shot_seg + (size_t)grp * K * SHOT_LDS_WORDS;
    ShotConsts k = shot_consts(dt);
    V3 tg = v3(target[i], target[n + i], target[2 * n + i]);
    const int nseg = (ticks + K - 1) / K;
    ShotState<float> s;
    int last_extra;
    shot_ckpt_load(ckpt + (size_t)(nseg - 1) * SHOT_CKPT_WORDS * n, n, i, s, last_extra);
    uint32_t fl = 0;
    for (int t = (nseg - 1) * K; t < ticks; t++) shot_step(s, shot_ctrl(ctrl, n, i, t), t, last_extra, fl, k);
    float g[SHOT_STATE_WORDS];
    shot_loss_grad(s, tg, dloss[i], g);
    float mine = 0.f;
    for (int sg = nseg - 1; sg >= 0; sg--) {
        const int t0 = sg * K, t1 = t0 + K < ticks ? t0 + K : ticks;
        ShotState<float> x;
        int lx;
        shot_ckpt_load(ckpt + (size_t)sg * SHOT_CKPT_WORDS * n, n, i, x, lx);
        for (int t = t0; t < t1; t++) {
            if (lane == 0) {
                float* r = seg + (t - t0) * SHOT_LDS_WORDS;
                for (int w = 0; w < SHOT_STATE_WORDS; w++) r[w] = shot_word(x, w);
                r[SHOT_STATE_WORDS] = __int_as_float(lx);
            }
            shot_step(x, shot_ctrl(ctrl, n, i, t), t, lx, fl, k);
        }
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
        for (int t = t1 - 1; t >= t0; t--) {
            const float* r = seg + (t - t0) * SHOT_LDS_WORDS;
            ShotState<float> st;
            for (int w = 0; w < SHOT_STATE_WORDS; w++) shot_word(st, w) = r[w];
            const int le = __float_as_int(r[SHOT_STATE_WORDS]);
            mine = shot_vjp_entry(st, shot_ctrl(ctrl, n, i, t), t, le, k, g, lane);
            for (int w = 0; w < SHOT_STATE_WORDS; w++) g[w] = __shfl(mine, w, SHOT_GROUP);
            if (lane >= SHOT_STATE_WORDS && lane < SHOT_INPUTS)
                dctrl[(size_t)t * 4 * n + (size_t)(lane - SHOT_STATE_WORDS) * n + i] = mine;
        }
        // the next segment's states overwrite this one's
        __builtin_amdgcn_fence(__ATOMIC_SEQ_CST, "workgroup");
        __builtin_amdgcn_wave_barrier();
    }
    if (ds0 && lane < SHOT_STATE_WORDS) ds0[(size_t)lane * n + i] = mine * shot_unit(lane);
}

// Backward with every tick's state at hand (K = 1): `per` pairs a wave, a lane
// each, take the ticks without a contact by the hand-written adjoint; where a
// pair has a contact, which is some ticks of a shot, 32 lanes take its 26
// tangents, two pairs at a time.
//
// What bounds it: the chain of ticks, 2.5 us each (16384 pairs: 78 % of a
// wave's cycles issue VALU instructions, it waits 14 %).  One group of lanes a pair
// ran all 26 tangents on every tick: 16384 pairs x 90 ticks 3210 us against 614,
// 101 x 60 298 against 186.
__global__ void __launch_bounds__(64) rsg_shot_backward_kept_kernel(int n, int ticks, int per, float dt,
                                                                    const float* ctrl, const float* target,
                                                                    const float* ckpt, const float* dloss,
                                                                    float* dctrl, float* ds0) {
    const int lane = threadIdx.x, first = blockIdx.x * per;
    const bool on = lane < per && first + lane < n;
    const int i = on ? first + lane : first;   // a lane without a pair reads the wave's first
    const ShotConsts k = shot_consts(dt);
    auto load = [&](int t, int at, ShotState<float>& s, int& le) {
        shot_ckpt_load(ckpt + (size_t)t * SHOT_CKPT_WORDS * n, n, at, s, le);
    };
    ShotState<float> x;
    int le;
    load(ticks - 1, i, x, le);
    ShotCtrl<float> c = shot_ctrl(ctrl, n, i, ticks - 1);
    float g[SHOT_STATE_WORDS];
    {
        ShotState<float> s = x;
        int last_extra = le;
        uint32_t fl = 0;
        shot_step(s, c, ticks - 1, last_extra, fl, k);
        shot_loss_grad(s, v3(target[i], target[n + i], target[2 * n + i]), dloss[i], g);
    }
    RSG_UNROLL_1
    for (int t = ticks - 1; t >= 0; t--) {
        const int before = t > 0 ? t - 1 : 0;
        ShotState<float> xb;
        int leb;
        load(before, i, xb, leb);
        const ShotCtrl<float> cb = shot_ctrl(ctrl, n, i, before);
        const bool touch = shot_touches(x, k);
        uint64_t touching = __ballot(on && touch);
        RSG_UNROLL_1
        while (touching) {
            const int a = __builtin_ctzll(touching);
            touching &= touching - 1u;
            const int b = touching ? __builtin_ctzll(touching) : a;
            touching &= touching - 1u;
            const int from = lane < SHOT_GROUP ? a : b, j = lane & (SHOT_GROUP - 1);
            ShotState<float> s;
            int last_extra;
            load(t, first + from, s, last_extra);
            float gs[SHOT_STATE_WORDS];
            for (int w = 0; w < SHOT_STATE_WORDS; w++) gs[w] = __shfl(g[w], from);
            const float mine = shot_vjp_entry(s, shot_ctrl(ctrl, n, first + from, t), t, last_extra, k, gs, j);
            if (j >= SHOT_STATE_WORDS && j < SHOT_INPUTS)
                dctrl[(size_t)t * 4 * n + (size_t)(j - SHOT_STATE_WORDS) * n + first + from] = mine;
            for (int w = 0; w < SHOT_STATE_WORDS; w++) {
                const float v = __shfl(mine, w + (lane == a ? 0 : SHOT_GROUP));
                g[w] = lane == a || lane == b ? v : g[w];
            }
        }
        if (on && !touch) {
            AirCtrl gc;
            shot_flight_vjp(x, c, k, g, gc);
            float* o = dctrl + (size_t)t * 4 * n;
            o[i] = gc.pitch; o[n + i] = gc.yaw; o[2 * n + i] = gc.roll; o[3 * n + i] = gc.boost;
        }
        x = xb;
        le = leb;
        c = cb;
    }
    if (ds0 && on)
        for (int w = 0; w < SHOT_STATE_WORDS; w++) ds0[(size_t)w * n + i] = g[w] * shot_unit(w);
}

namespace rsg {

// 64-lane workgroups spread the cars over every CU.
hipError_t launch_air_forward(bool rows, int n, int ticks, int K, float dt, const float* s0, const float* ctrl,
                              const float* target, float* s_out, float* loss, float* ckpt, float* kept,
                              float* kept_target, hipStream_t s) {
    const int block = 64, grid = (n + block - 1) / block;
    hipLaunchKernelGGL(rows ? rsg_air_forward_kernel<true> : rsg_air_forward_kernel<false>, dim3(grid), dim3(block), 0, s,
                       n, ticks, K, dt, s0, ctrl, target, s_out, loss, ckpt, kept, kept_target);
    return hipGetLastError();
}

hipError_t launch_air_backward(bool rows, int n, int ticks, int K, float dt, const float* ctrl, const float* target,
                               const float* ckpt, const float* dloss, float* dctrl, float* ds0, hipStream_t s) {
    const int block = 64, grid = (n + block - 1) / block;
    if (K == 1)
        hipLaunchKernelGGL(rows ? rsg_air_backward_kept_kernel<true> : rsg_air_backward_kept_kernel<false>, dim3(grid),
                           dim3(block), 0, s, n, ticks, dt, ctrl, target, ckpt, dloss, dctrl, ds0);
    else
        hipLaunchKernelGGL(rows ? rsg_air_backward_kernel<true> : rsg_air_backward_kernel<false>, dim3(grid), dim3(block),
                           0, s, n, ticks, K, dt, ctrl, target, ckpt, dloss, dctrl, ds0);
    return hipGetLastError();
}

// Pairs per wave: spread over the SIMDs first, as a wave takes the contact path
// on every tick on which one of its pairs has a contact (forward, 16384 pairs x
// 90 ticks: 301 us at 16 a wave against 375 at 64; 101 x 60: 117 at 1 against
// 291).  (A wave holds any number, so the count of an MI355X serves elsewhere.)
static int shot_per_wave(int n) {
    constexpr int SIMDS = 1024;
    const int per = (n + SIMDS - 1) / SIMDS;
    return per > 64 ? 64 : per;
}

hipError_t launch_shot_forward(int n, int ticks, int K, float dt, const float* state0, const float* ctrl,
                               const float* target, float* state_out, float* loss, float* ckpt, uint32_t* flags,
                               hipStream_t s) {
    const int block = shot_per_wave(n), grid = (n + block - 1) / block;
    hipLaunchKernelGGL(rsg_shot_forward_kernel, dim3(grid), dim3(block), 0, s, n, ticks, K, dt, state0, ctrl, target,
                       state_out, loss, ckpt, flags);
    return hipGetLastError();
}

hipError_t launch_shot_backward(int n, int ticks, int K, float dt, const float* ctrl, const float* target,
                                const float* ckpt, const float* dloss, float* dctrl, float* ds0, hipStream_t s) {
    if (K == 1) {
        const int per = shot_per_wave(n);
        hipLaunchKernelGGL(rsg_shot_backward_kept_kernel, dim3((n + per - 1) / per), dim3(64), 0, s, n, ticks, per, dt, ctrl,
                           target, ckpt, dloss, dctrl, ds0);
        return hipGetLastError();
    }
    const int block = 256, per_block = block / SHOT_GROUP, grid = (n + per_block - 1) / per_block;
    const size_t lds = (size_t)per_block * K * SHOT_LDS_WORDS * sizeof(float);
    hipLaunchKernelGGL(rsg_shot_backward_kernel, dim3(grid), dim3(block), lds, s, n, ticks, K, dt, ctrl, target, ckpt,
                       dloss, dctrl, ds0);
    return hipGetLastError();
}

}  // namespace rsg
