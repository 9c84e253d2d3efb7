// rsg_torch.cpp -- LibTorch C++ autograd Functions over the differentiable
// rollouts of librsg.so (rsg_air_rollout / rsg_air_rollout_backward and
// rsg_shot_rollout / rsg_shot_rollout_backward, include/rsg.h), built as the
// Python extension module rsg_torch.
//
//   loss, final = rsg_torch.air_rollout(state0, controls, target, ckpt_every, tick_rate, stream)
//
// state0 [n, 13] (position uu, quaternion x y z w, velocity uu/s, angular
// velocity rad/s), controls [ticks, n, 4] (pitch, yaw, roll in [-1, 1], boost
// in [0, 1]), target [n, 7] (quaternion, position uu); GPU tensors.  The
// forward keeps a checkpoint of every car's state every ckpt_every ticks (None:
// chosen by size, chosen_every below); the backward recomputes each segment
// from its checkpoint and runs the hand-written adjoint kernel.  Gradients flow
// to controls and state0.
// `stream` is the hipStream_t to run on (the caller's current stream); the
// backward runs on the stream of its forward, as autograd does for every op.
#include <optional>

#include <torch/extension.h>

#include <string>

#include "rsg.h"

namespace {

void check(int rc, const char* what) {
    TORCH_CHECK(rc >= 0, what, ": ", rsg_last_error());
}

using torch::autograd::AutogradContext;
using torch::autograd::variable_list;

// Ticks per checkpoint where the caller names none: every tick's state, which
// the backward pass then need not compute again, up to KEEP_BYTES of them
// (65536 cars x 120 ticks, 409 MB: 455 us in all against 548 at one every 16;
// 16384 shots x 90 ticks, 136 MB: 950 us against 3540); past it one state every
// CKPT_EVERY ticks, as the states would crowd out a caller's own memory.
constexpr int64_t KEEP_BYTES = (int64_t)512 << 20;
constexpr int64_t CKPT_EVERY = 16, MAX_CKPT_EVERY = 32;
constexpr int64_t AIR_WORDS = 13, SHOT_WORDS = 23;   // of a checkpoint
int64_t chosen_every(int64_t n, int64_t ticks, int64_t words) {
    return n * ticks * words * (int64_t)sizeof(float) <= KEEP_BYTES ? 1 : CKPT_EVERY;
}
int64_t air_ckpt_every(int64_t n, int64_t ticks) { return chosen_every(n, ticks, AIR_WORDS); }
int64_t shot_ckpt_every(int64_t n, int64_t ticks) { return chosen_every(n, ticks, SHOT_WORDS); }

// Whether a rollout of these inputs records a graph (the test that
// Function::apply makes).  One that does not has no backward pass to keep
// states and copies for (65536 cars x 120 ticks under no_grad: 99 us and 4 MB
// against 175 us and 539 MB; 16384 shots x 90 ticks: 296 against 313).
bool records_graph(const torch::Tensor& state0, const torch::Tensor& controls, const torch::Tensor& target) {
    return torch::GradMode::is_enabled() &&
           (state0.requires_grad() || controls.requires_grad() || target.requires_grad());
}

struct AirRolloutFn : public torch::autograd::Function<AirRolloutFn> {
    static variable_list forward(AutogradContext* ctx, torch::Tensor state0, torch::Tensor controls,
                                 torch::Tensor target, int64_t ckpt_every, double tick_rate, int64_t stream,
                                 bool graph = true) {
        TORCH_CHECK(state0.is_cuda() && controls.is_cuda() && target.is_cuda(),
                    "air_rollout: tensors must be on the GPU (the kernels are HIP only)");
        TORCH_CHECK(state0.dim() == 2 && state0.size(1) == 13, "air_rollout: state0 must be [n, 13]");
        TORCH_CHECK(controls.dim() == 3 && controls.size(2) == 4 && controls.size(1) == state0.size(0),
                    "air_rollout: controls must be [ticks, n, 4]");
        TORCH_CHECK(target.dim() == 2 && target.size(1) == 7 && target.size(0) == state0.size(0),
                    "air_rollout: target must be [n, 7]");
        const int64_t n = state0.size(0), ticks = controls.size(0);
        auto s0 = state0.to(torch::kFloat).contiguous();
        auto ctrl = controls.to(torch::kFloat).contiguous();
        auto tgt = target.to(torch::kFloat).contiguous();
        const int64_t nseg = (ticks + ckpt_every - 1) / ckpt_every;
        auto opts = s0.options();
        // the states, and the backward pass's own copies, as the caller may change its tensors
        torch::Tensor ckpt, kept, kept_target;
        if (graph) ckpt = torch::empty({nseg * AIR_WORDS * n}, opts);
        auto out = torch::empty({n, 13}, opts);
        auto loss = torch::empty({n}, opts);
        if (graph) {
            kept = torch::empty_like(ctrl);
            kept_target = torch::empty_like(tgt);
        }
        auto data = [](const torch::Tensor& t) { return t.defined() ? t.data_ptr<float>() : nullptr; };
        check(rsg_air_rollout_rows((int)n, (int)ticks, (int)ckpt_every, (float)tick_rate, s0.data_ptr<float>(),
                                   ctrl.data_ptr<float>(), tgt.data_ptr<float>(), out.data_ptr<float>(),
                                   loss.data_ptr<float>(), data(ckpt), data(kept), data(kept_target), (void*)stream),
              "rsg_air_rollout");
        if (graph) ctx->save_for_backward({kept, kept_target, ckpt});
        ctx->saved_data["n"] = n;
        ctx->saved_data["ticks"] = ticks;
        ctx->saved_data["ckpt_every"] = ckpt_every;
        ctx->saved_data["tick_rate"] = tick_rate;
        ctx->saved_data["stream"] = stream;
        ctx->mark_non_differentiable({out});
        return {loss, out};
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        auto saved = ctx->get_saved_variables();
        auto ctrl = saved[0], tgt = saved[1], ckpt = saved[2];
        const int64_t n = ctx->saved_data["n"].toInt(), ticks = ctx->saved_data["ticks"].toInt();
        const int64_t ckpt_every = ctx->saved_data["ckpt_every"].toInt();
        const double tick_rate = ctx->saved_data["tick_rate"].toDouble();
        const int64_t stream = ctx->saved_data["stream"].toInt();
        auto dl = grads[0].defined() ? grads[0].to(torch::kFloat).contiguous() : torch::zeros({n}, ctrl.options());
        auto dctrl = torch::empty_like(ctrl);
        auto ds0 = torch::empty({n, 13}, ctrl.options());
        check(rsg_air_rollout_rows_backward((int)n, (int)ticks, (int)ckpt_every, (float)tick_rate,
                                            ctrl.data_ptr<float>(), tgt.data_ptr<float>(), ckpt.data_ptr<float>(),
                                            dl.data_ptr<float>(), dctrl.data_ptr<float>(), ds0.data_ptr<float>(),
                                            (void*)stream),
              "rsg_air_rollout_backward");
        return {ds0, dctrl, torch::Tensor(), torch::Tensor(), torch::Tensor(), torch::Tensor(),
                torch::Tensor()};
    }
};

// The aerial shot (rsg_shot_rollout / rsg_shot_rollout_backward): state0
// [n, 22], controls [ticks, n, 4], target [n, 3]; returns loss [n], the final
// state [n, 22] and the contact flags [n] (int32).
struct ShotRolloutFn : public torch::autograd::Function<ShotRolloutFn> {
    static variable_list forward(AutogradContext* ctx, torch::Tensor state0, torch::Tensor controls,
                                 torch::Tensor target, int64_t ckpt_every, double tick_rate, int64_t stream,
                                 bool graph = true) {
        TORCH_CHECK(state0.is_cuda() && controls.is_cuda() && target.is_cuda(),
                    "shot_rollout: tensors must be on the GPU (the kernels are HIP only)");
        TORCH_CHECK(state0.dim() == 2 && state0.size(1) == 22, "shot_rollout: state0 must be [n, 22]");
        TORCH_CHECK(controls.dim() == 3 && controls.size(2) == 4 && controls.size(1) == state0.size(0),
                    "shot_rollout: controls must be [ticks, n, 4]");
        TORCH_CHECK(target.dim() == 2 && target.size(1) == 3 && target.size(0) == state0.size(0),
                    "shot_rollout: target must be [n, 3]");
        const int64_t n = state0.size(0), ticks = controls.size(0);
        auto s0 = state0.to(torch::kFloat).t().contiguous();
        auto ctrl = controls.to(torch::kFloat).permute({0, 2, 1}).contiguous();
        auto tgt = target.to(torch::kFloat).t().contiguous();
        const int64_t nseg = (ticks + ckpt_every - 1) / ckpt_every;
        auto opts = s0.options();
        auto ckpt = torch::empty({nseg * SHOT_WORDS * n}, opts);
        auto out = torch::empty({22, n}, opts);
        auto loss = torch::empty({n}, opts);
        auto flags = torch::empty({n}, opts.dtype(torch::kInt32));
        check(rsg_shot_rollout((int)n, (int)ticks, (int)ckpt_every, (float)tick_rate, s0.data_ptr<float>(),
                               ctrl.data_ptr<float>(), tgt.data_ptr<float>(), out.data_ptr<float>(),
                               loss.data_ptr<float>(), ckpt.data_ptr<float>(),
                               reinterpret_cast<uint32_t*>(flags.data_ptr<int32_t>()), (void*)stream),
              "rsg_shot_rollout");
        if (graph) ctx->save_for_backward({ctrl, tgt, ckpt});
        ctx->saved_data["n"] = n;
        ctx->saved_data["ticks"] = ticks;
        ctx->saved_data["ckpt_every"] = ckpt_every;
        ctx->saved_data["tick_rate"] = tick_rate;
        ctx->saved_data["stream"] = stream;
        auto final_state = out.t().contiguous();
        ctx->mark_non_differentiable({final_state, flags});
        return {loss, final_state, flags};
    }

    static variable_list backward(AutogradContext* ctx, variable_list grads) {
        auto saved = ctx->get_saved_variables();
        auto ctrl = saved[0], tgt = saved[1], ckpt = saved[2];
        const int64_t n = ctx->saved_data["n"].toInt(), ticks = ctx->saved_data["ticks"].toInt();
        const int64_t ckpt_every = ctx->saved_data["ckpt_every"].toInt();
        const double tick_rate = ctx->saved_data["tick_rate"].toDouble();
        const int64_t stream = ctx->saved_data["stream"].toInt();
        auto dl = grads[0].defined() ? grads[0].to(torch::kFloat).contiguous() : torch::zeros({n}, ctrl.options());
        auto dctrl = torch::empty_like(ctrl);
        auto ds0 = torch::empty({22, n}, ctrl.options());
        check(rsg_shot_rollout_backward((int)n, (int)ticks, (int)ckpt_every, (float)tick_rate, ctrl.data_ptr<float>(),
                                        tgt.data_ptr<float>(), ckpt.data_ptr<float>(), dl.data_ptr<float>(),
                                        dctrl.data_ptr<float>(), ds0.data_ptr<float>(), (void*)stream),
              "rsg_shot_rollout_backward");
        return {ds0.t().contiguous(), dctrl.permute({0, 2, 1}).contiguous(), torch::Tensor(), torch::Tensor(),
                torch::Tensor(), torch::Tensor(), torch::Tensor()};
    }
};

std::vector<torch::Tensor> shot_rollout(torch::Tensor state0, torch::Tensor controls, torch::Tensor target,
                                        std::optional<int64_t> ckpt_every, double tick_rate, int64_t stream) {
    TORCH_CHECK(!ckpt_every || (*ckpt_every >= 1 && *ckpt_every <= MAX_CKPT_EVERY),
                "shot_rollout: ckpt_every must be within [1, 32]");
    // (without a graph its checkpoints go unused: few; tensors of other shapes
    // are refused by the Function)
    const bool graph = records_graph(state0, controls, target);
    const int64_t every = ckpt_every ? *ckpt_every
                        : graph && controls.dim() == 3 ? shot_ckpt_every(controls.size(1), controls.size(0)) : CKPT_EVERY;
    auto r = ShotRolloutFn::apply(state0, controls, target, every, tick_rate, stream, graph);
    return {r[0], r[1], r[2]};
}

std::vector<torch::Tensor> air_rollout(torch::Tensor state0, torch::Tensor controls, torch::Tensor target,
                                       std::optional<int64_t> ckpt_every, double tick_rate, int64_t stream) {
    TORCH_CHECK(!ckpt_every || (*ckpt_every >= 1 && *ckpt_every <= MAX_CKPT_EVERY),
                "air_rollout: ckpt_every must be within [1, 32]");
    // (tensors of other shapes are refused by the Function)
    // (tensors of other shapes are refused by the Function)
    const bool graph = records_graph(state0, controls, target);
    const int64_t every = ckpt_every ? *ckpt_every
                        : controls.dim() == 3 ? air_ckpt_every(controls.size(1), controls.size(0)) : CKPT_EVERY;
    auto r = AirRolloutFn::apply(state0, controls, target, every, tick_rate, stream, graph);
    return {r[0], r[1]};
}

}  // namespace

PYBIND11_MODULE(rsg_torch, m) {
    m.doc() = "LibTorch autograd Function over the differentiable air-control rollout of librsg.so";
    m.def("air_rollout", &air_rollout, "loss, final = air_rollout(state0, controls, target, ckpt_every, tick_rate, stream)",
          pybind11::arg("state0"), pybind11::arg("controls"), pybind11::arg("target"), pybind11::arg("ckpt_every"),
          pybind11::arg("tick_rate"), pybind11::arg("stream"));
    m.def("air_ckpt_every", &air_ckpt_every, "Ticks per checkpoint of air_rollout with ckpt_every=None",
          pybind11::arg("n"), pybind11::arg("ticks"));
    m.def("shot_ckpt_every", &shot_ckpt_every, "Ticks per checkpoint of shot_rollout with ckpt_every=None",
          pybind11::arg("n"), pybind11::arg("ticks"));
    m.def("shot_rollout", &shot_rollout,
          "loss, final, flags = shot_rollout(state0, controls, target, ckpt_every, tick_rate, stream)",
          pybind11::arg("state0"), pybind11::arg("controls"), pybind11::arg("target"), pybind11::arg("ckpt_every"),
          pybind11::arg("tick_rate"), pybind11::arg("stream"));
}
