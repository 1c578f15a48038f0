"""Masks given as bool: the ops take them as bytes of their own, laid out one
after the other, as they were at the call."""
import pytest
import torch

from dreamplace_amd import _native as N


@pytest.mark.parametrize("kind", ["plain", "strided", "expanded"])
def test_bytes(kind):
    b = torch.tensor([True, False, False, True, True, False])
    m = {"plain": b, "strided": b[::2], "expanded": b[:1].expand(6)}[kind]
    u = N.as_u8(m)
    want = m.tolist()
    assert u.dtype == torch.uint8 and u.is_contiguous() and u.tolist() == want
    b.logical_not_()
    assert u.tolist() == want
    assert N.as_u8(None) is None and N.as_u8(u) is u


@pytest.mark.gpu
def test_strided_mask(gpu):
    from dreamplace_amd.hpwl import hpwl_fp64
    print("case strided net mask", flush=True)
    pos = torch.rand(40, device=gpu)
    flat, start = torch.arange(20, device=gpu).int(), torch.arange(0, 21, 4, device=gpu).int()
    both = torch.tensor([[True, False], [False, False], [True, True], [False, True], [True, False]],
                        device=gpu)
    for m in (both[:, 0], both[2:3, 0].expand(5)):
        args = pos, flat, start, torch.ones(5, device=gpu)
        assert torch.equal(hpwl_fp64(*args, m), hpwl_fp64(*args, m.clone().contiguous()))


@pytest.mark.gpu
@pytest.mark.parametrize("model", ["wa", "lse"])
def test_mask_changed_after_forward(gpu, model):
    """The backward takes the pin mask that the forward was given."""
    from dreamplace_amd.logsumexp_wirelength import LogSumExpWirelength
    from dreamplace_amd.weighted_average_wirelength import WeightedAverageWirelength
    print("case mask after forward %s" % model, flush=True)
    op = WeightedAverageWirelength if model == "wa" else LogSumExpWirelength
    flat, start = torch.arange(20, device=gpu).int(), torch.arange(0, 21, 4, device=gpu).int()
    mask = torch.arange(20, device=gpu) % 3 == 0
    f = op(flat, start, flat // 4, torch.ones(5, device=gpu), torch.ones(5, device=gpu).bool(),
           mask, torch.tensor(0.5, device=gpu), algorithm="merged")
    pos = torch.rand(40, device=gpu, generator=torch.Generator(device=gpu).manual_seed(1))
    pos.requires_grad_(True)
    want = torch.autograd.grad(f(pos), [pos])[0]
    assert bool((want[:20][mask] == 0).all()) and bool((want[:20][~mask] != 0).all())
    out = f(pos)
    mask.logical_not_()
    assert torch.equal(torch.autograd.grad(out, [pos])[0], want)
