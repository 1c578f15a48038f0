"""Nets of more than 64 pins through the exchange in LDS tiles (k_wa_big on its
places), among other nets and with no other net at all: an evaluation against
one through the slices.  The same arithmetic per net and per node, so the
derivatives and the per-net lengths are equal; the totals add the same FP64
terms, none negative, in another order: at most 32 additions in a row on either
side, and one rounding to the data type."""
import numpy as np
import pytest
import torch

from _util import design
from dreamplace_amd import engine, synth

pytestmark = pytest.mark.gpu


def regrouped(d, degrees):
    """Design `d` with its pins, in their order, in nets of these degrees."""
    d = synth.Design(d)
    deg = np.asarray(degrees)
    E, rng = len(deg), np.random.default_rng(7)
    assert deg.sum() == d.num_pins
    d.update(num_nets=E, pin2net_map=np.repeat(np.arange(E, dtype=np.int32), deg),
             flat_net2pin_start_map=np.concatenate([[0], np.cumsum(deg)]).astype(np.int32),
             net_weights=(0.5 + rng.random(E)).astype(d.pos.dtype),
             net_mask_all=np.ones(E, np.uint8),
             net_mask_ignore_large_degrees=(rng.random(E) < 0.9).astype(np.uint8))
    return d


def degrees(kind, P):
    if kind == "only":  # the last net takes what is left
        n = P // 100
        return [100] * (n - 1) + [P - 100 * (n - 1)]
    rng = np.random.default_rng(8)
    deg = []
    while sum(deg) < P - 6000:
        deg += list(rng.integers(1, 9, 400)) + [64, 65, int(rng.integers(66, 2500))]
    return deg + [P - sum(deg)]


@pytest.mark.parametrize("kind", ["only", "among"])
@pytest.mark.parametrize("model", ["wa", "centred", "lse"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64], ids=["f32", "f64"])
def test_big_nets(gpu, monkeypatch, dtype, model, kind):
    from dreamplace_amd.engine import DeviceDesign, PlacementObjective
    print("case big nets in tiles %s %s %s" % (np.dtype(dtype).name, model, kind), flush=True)
    d = design(1, scale=0.01, dtype=dtype)
    d = regrouped(d, degrees(kind, d.num_pins))
    dd = DeviceDesign(d, gpu)
    kw = dict(wirelength="logsumexp") if model == "lse" else dict(
        wa_arith="centred" if model == "centred" else "reference")
    res = []
    for least in (1, 1 << 40):
        monkeypatch.setattr(engine, "TILE_MIN_PINS", least)
        obj = PlacementObjective(dd, d.wa_gamma, density_weight=0.2, algorithm="tiled",
                                 precision="fp64" if dtype is np.float64 else "fp32",
                                 schedule="pins", track_metrics=True, **kw)
        plan = obj.pin_plan
        assert (plan.tiles is not None) == (least == 1) and plan.num_big > 0
        if least == 1:
            assert (len(plan.tiles["net_tiles"]) == 1) == (kind == "only")
        plan.ws.fill_(255)  # what no kernel writes is not a number
        f, g = obj.evaluate(dd.pos)
        res.append([g.clone(), obj.net_hpwl.clone(), obj.wl.clone(), f.clone()])
    a, b = res
    assert torch.equal(a[0], b[0]) and torch.equal(a[1], b[1])
    eps = torch.finfo(dd.dtype).eps + 64 * 2.0 ** -53
    assert abs(float(a[2] - b[2])) <= eps * float(b[2])
    # the objective adds one product and one sum in the data type to that
    assert abs(float(a[3] - b[3])) <= 2 * eps * (abs(float(b[2])) + abs(float(b[3])))
