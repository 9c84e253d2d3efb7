"""ckpt_every of the differentiable rollouts: an explicit value bounds the states
that a graph holds until its backward pass, one left out is chosen by size, and
values out of range are refused."""
import pytest
import torch


def test_chosen_by_size():
    from rocketsim_amd.adjoint import air_ckpt_every, shot_ckpt_every
    mb = 1 << 20
    for every, words in ((air_ckpt_every, 13), (shot_ckpt_every, 23)):
        most = 512 * mb // (4 * words * 100)    # cars whose 100 states each take up to 512 MB
        assert every(most, 100) == 1
        assert every(most + 1, 100) == 16
        assert every(1, 1) == 1


def _inputs(kind, n, ticks):
    g = torch.Generator().manual_seed(n)
    s0 = torch.randn(n, 13 if kind == "air" else 22, generator=g)
    s0[:, :3] += 500.0
    s0[:, 3:7] = torch.nn.functional.normalize(s0[:, 3:7], dim=-1)
    ctrl = torch.tanh(torch.randn(ticks, n, 4, generator=g)).abs()
    tgt = torch.randn(n, 7 if kind == "air" else 3, generator=g)
    return s0.cuda(), ctrl.cuda().requires_grad_(True), tgt.cuda()


@pytest.mark.gpu
@pytest.mark.parametrize("kind,words", [("air", 13), ("shot", 23)])
def test_the_graph_holds_a_state_every_ckpt_every_ticks(kind, words):
    from rocketsim_amd import adjoint
    fn = getattr(adjoint, kind + "_rollout")
    n, ticks = 3000, 70
    s0, ctrl, tgt = _inputs(kind, n, ticks)

    def held(**kw):
        torch.cuda.synchronize()
        before = torch.cuda.memory_allocated()
        out = fn(s0, ctrl, tgt, **kw)
        return torch.cuda.memory_allocated() - before, out

    held()          # first use
    state = 4 * words * n
    # what it holds whatever the distance: outputs, the controls' and the
    # target's copies (each allocation is rounded up to at most 512 bytes more)
    other = held(ckpt_every=1)[0] - ticks * state
    for every, segments in ((None, 70), (1, 70), (3, 24), (16, 5), (32, 3)):
        got, _ = held(ckpt_every=every) if every else held()
        assert abs(got - other - segments * state) <= 1024, (every, got)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["air", "shot"])
@pytest.mark.parametrize("every", [0, -1, 33])
def test_out_of_range_is_refused(kind, every):
    from rocketsim_amd import adjoint
    with pytest.raises(RuntimeError, match="ckpt_every"):
        getattr(adjoint, kind + "_rollout")(*_inputs(kind, 5, 4), ckpt_every=every)
