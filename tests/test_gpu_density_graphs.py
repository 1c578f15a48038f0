"""The density op's forward and backward captured as two graphs, as
torch.cuda.make_graphed_callables does, with calls on the op between replays:
the gradient is that of the captured positions."""
import pytest
import torch

from _util import design, to_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("arithmetic", ["reference", "bin_relative"])
def test_two_graphs(gpu, monkeypatch, arithmetic):
    from dreamplace_amd import electric_overflow
    from dreamplace_amd.electric_potential import ElectricPotential
    print("case density graphs %s" % arithmetic, flush=True)
    monkeypatch.setattr(electric_overflow, "TILED_MIN_CELLS", 1)
    d = design(1, scale=0.002)
    t = to_dev(d, gpu)
    op = ElectricPotential(
        t["node_size_x"], t["node_size_y"], t["bin_center_x"], t["bin_center_y"],
        d.target_density, d.xl, d.yl, d.xh, d.yh, d.bin_size_x, d.bin_size_y,
        d.num_movable_nodes, d.num_terminals, d.num_filler_nodes, 0, True, t["sorted_node_map"],
        movable_macro_mask=t["movable_macro_mask"], arithmetic=arithmetic)

    def both(p):
        p = p.clone().requires_grad_(True)
        return torch.autograd.grad(op(p), [p])[0]

    positions = [t["pos"] + k * d.bin_size_x for k in (0.0, 0.75, 1.5, 2.25)]
    want = [both(p) for p in positions]
    pos = positions[0].clone().requires_grad_(True)
    one = torch.ones((), dtype=pos.dtype, device=gpu)
    torch.cuda.synchronize()
    forward, backward = torch.cuda.CUDAGraph(), torch.cuda.CUDAGraph()
    with torch.cuda.graph(forward):
        energy = op(pos)
    with torch.cuda.graph(backward, pool=forward.pool()):
        grad = torch.autograd.grad(energy, [pos], [one])[0]
    for k in (1, 2, 3):
        with torch.no_grad():
            pos.copy_(positions[k])
        forward.replay()
        assert torch.equal(both(positions[k - 1]), want[k - 1])
        backward.replay()
        torch.cuda.synchronize()
        assert torch.equal(grad, want[k])
