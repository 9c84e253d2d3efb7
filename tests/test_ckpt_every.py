"""ckpt_every of the differentiable rollouts: an explicit value bounds the states
that a graph holds until its backward pass, one left out is chosen by size, and
values out of range are refused; a rollout that records no graph keeps none."""
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

    def saved(**kw):
        sizes = []
        with torch.autograd.graph.saved_tensors_hooks(lambda x: sizes.append(x.numel()) or x, lambda x: x):
            fn(s0, ctrl, tgt, **kw)
        return sizes

    for every, segments in ((None, 70), (1, 70), (3, 24), (16, 5), (32, 3)):
        got = saved(ckpt_every=every) if every else saved()
        assert sorted(got) == sorted([ctrl.numel(), tgt.numel(), segments * words * n]), every


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["air", "shot"])
@pytest.mark.parametrize("every", [0, -1, 33])
def test_out_of_range_is_refused(kind, every):
    from rocketsim_amd import adjoint
    with pytest.raises(RuntimeError, match="ckpt_every"):
        getattr(adjoint, kind + "_rollout")(*_inputs(kind, 5, 4), ckpt_every=every)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["air", "shot"])
@pytest.mark.parametrize("off", ["no_grad", "inference_mode", "no input requires grad"])
def test_no_states_are_kept_without_a_graph(kind, off):
    from rocketsim_amd import adjoint
    fn = getattr(adjoint, kind + "_rollout")
    n, ticks = 3000, 70
    s0, ctrl, tgt = _inputs(kind, n, ticks)
    want = fn(s0, ctrl, tgt)
    if off == "no input requires grad":
        ctrl = ctrl.detach()
        run = lambda: fn(s0, ctrl, tgt)                     # noqa: E731
    else:
        run = getattr(torch, off)()(lambda: fn(s0, ctrl, tgt))
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    got = run()
    peak = torch.cuda.max_memory_allocated() - before
    for a, b in zip(got, want):
        assert not a.requires_grad and torch.equal(a, b.detach())
    # outputs alone; the shot has transposed inputs and outputs and 5 states
    # besides.  (The allocator leaves up to 512 bytes unused of a block up to
    # 1 MB, and up to 1 MB of a larger one; the shot has two of these.)
    words = 14 if kind == "air" else 22 + ticks * 4 + 3 + 22 * 2 + 2 + 5 * 23
    spare = 7 * 512 + (0 if kind == "air" else 2 << 20)
    assert peak <= 4 * words * n + spare, (peak, 4 * words * n)


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["air", "shot"])
def test_a_graph_through_the_target_alone(kind):
    """The target takes no gradient; the backward pass runs all the same."""
    from rocketsim_amd import adjoint
    s0, ctrl, tgt = _inputs(kind, 5, 4)
    tgt.requires_grad_(True)
    loss = getattr(adjoint, kind + "_rollout")(s0, ctrl.detach(), tgt)[0]
    assert loss.requires_grad
    got, = torch.autograd.grad(loss.sum(), [tgt], allow_unused=True)
    assert got is None or not got.any()
