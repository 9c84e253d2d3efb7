"""The air rollout over arrays by car, with every tick's state kept, against
the one over arrays by word with checkpoints: the same bits, at tick counts
around the group of loads and the checkpoint distance, for one car, a ragged
wave and several, for inputs that are views at odd offsets or transposed, and
when the caller's tensors change between forward and backward."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _problem(n, ticks, seed):
    g = torch.Generator().manual_seed(seed)
    s0 = torch.cat([torch.randn(n, 3, generator=g) * 800, torch.nn.functional.normalize(torch.randn(n, 4, generator=g), dim=-1),
                    torch.randn(n, 3, generator=g) * 900, torch.randn(n, 3, generator=g) * 3], -1)
    ctrl = torch.cat([torch.tanh(torch.randn(ticks, n, 3, generator=g)), torch.rand(ticks, n, 1, generator=g)], -1)
    tgt = torch.cat([torch.nn.functional.normalize(torch.randn(n, 4, generator=g), dim=-1),
                     torch.randn(n, 3, generator=g) * 500], -1)
    return s0.cuda(), ctrl.cuda(), tgt.cuda()


def _grads(fn, s0, ctrl, tgt, change=False):
    s0, ctrl = s0.detach().requires_grad_(True), ctrl.detach().requires_grad_(True)
    loss, final = fn(s0, ctrl, tgt)
    if change:
        with torch.no_grad():
            ctrl.zero_()
            tgt.zero_()
    ds0, dctrl = torch.autograd.grad((loss * torch.arange(1, loss.numel() + 1, device="cuda")).sum(), [s0, ctrl])
    return [x.contiguous() for x in (loss, final, ds0, dctrl)]


@pytest.mark.parametrize("n,ticks", [(1, 1), (1, 4), (65, 3), (64, 5), (257, 17), (130, 33)])
def test_by_car_equals_by_word(n, ticks):
    from rocketsim_amd.adjoint import AirRollout, air_rollout
    s0, ctrl, tgt = _problem(n, ticks, n + ticks)
    want = _grads(lambda *a: AirRollout.apply(*a), s0, ctrl, tgt)

    def odd(x):     # the same values at an address off 16 bytes
        return torch.cat([torch.zeros(1, device="cuda"), x.flatten()])[1:].view(x.shape)

    def turned(x):  # ... with the last two dimensions' strides exchanged
        return x.transpose(-1, -2).contiguous().transpose(-1, -2)

    for make in (lambda x: x.clone(), odd, turned):
        for got, w in zip(_grads(air_rollout, make(s0), make(ctrl), make(tgt)), want):
            assert torch.equal(got, w)
    for got, w in zip(_grads(air_rollout, s0.clone(), ctrl.clone(), tgt.clone(), change=True), want):
        assert torch.equal(got, w)
