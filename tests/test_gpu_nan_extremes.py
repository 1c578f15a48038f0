"""A net's extent with pins that are not a number.  HPWL takes the first pin as
it is and each later one where it compares; the wirelength pass takes those
that compare.  Which lanes of a net hold them does not matter."""
import numpy as np
import pytest
import torch

from dreamplace_amd import _native as N

pytestmark = pytest.mark.gpu

DEGREES = [3, 4, 5, 6, 8, 9, 12, 16, 17, 24, 32, 33, 50, 64, 65, 100, 130]


def lanes(d):
    return 1 if d <= 4 else 2 if d <= 8 else 4 if d <= 16 else 8 if d <= 32 else 16 if d <= 64 else 64


def nets(first):
    """(x, y of the pins) of each degree: without one lane's pins, with only the
    first and the last pin of all, and (first) without the first pin."""
    rng = np.random.default_rng(5)
    for d in DEGREES:
        for lost in [range(lane, d, lanes(d)) for lane in range(lanes(d))] + [range(1, d - 1)]:
            v = rng.uniform(10, 90, (2, d))
            v[0, lost] = np.nan
            v[1, d - 1] = np.nan
            if first or not np.isnan(v[0, 0]):
                yield v


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
def test_hpwl(gpu, dtype):
    from dreamplace_amd.hpwl import hpwl_fp64
    print("case hpwl of pins not a number %s" % dtype, flush=True)
    for v in nets(True):
        p = torch.from_numpy(v).to(dtype)
        want = 0.0
        for c in p:
            lo = hi = c[0]
            for u in c[1:]:
                lo, hi = u if u < lo else lo, u if u > hi else hi
            want += float(hi - lo)
        d = p.shape[1]
        got = float(hpwl_fp64(p.reshape(-1).to(gpu), torch.arange(d, device=gpu).int(),
                              torch.tensor([0, d], device=gpu).int(), torch.ones(1, device=gpu, dtype=dtype),
                              torch.ones(1, device=gpu).byte()))
        assert (np.isnan(want) and np.isnan(got)) or abs(got - want) <= 1e-4, (d, got, want)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64], ids=["f32", "f64"])
@pytest.mark.parametrize("model", [N.DP_WL_WEIGHTED_AVERAGE, N.DP_WL_LOGSUMEXP,
                                   N.DP_WL_WEIGHTED_AVERAGE_CENTRED])
def test_slices(gpu, dtype, model):
    from dreamplace_amd.engine import pack_slices
    print("case slices of pins not a number %s %d" % (dtype, model), flush=True)
    vs = list(nets(False))
    deg = np.array([v.shape[1] for v in vs])
    E, P = len(deg), int(deg.sum())
    start = np.concatenate([[0], np.cumsum(deg)]).astype(np.int32)
    slices, lane_nets, big, slot, slots = pack_slices(start)
    up = lambda a, t=None: torch.from_numpy(np.ascontiguousarray(a)).to(gpu, t)
    pins, start_d = up(np.arange(P, dtype=np.int32)), up(start)
    p2net = up(np.repeat(np.arange(E, dtype=np.int32), deg))
    one = up(np.arange(P + 1, dtype=np.int32))  # a node for each pin
    pos, zero = up(np.concatenate(vs, 1).ravel(), dtype), torch.zeros(P, dtype=dtype, device=gpu)
    code, st = N.dtype_code(pos), N.stream_ptr(pos.device)
    ints = lambda n: torch.zeros(n, dtype=torch.int32, device=gpu)
    prep = torch.empty(N.query("dp_wa_prepare_workspace_bytes", P), dtype=torch.uint8, device=gpu)
    off, dst, node, meta = torch.zeros(2 * P, dtype=dtype, device=gpu), ints(P), ints(P), ints(slots)
    slot_d, sl, ln, bg = up(slot), up(slices), up(lane_nets), up(big)
    N.call("dp_wa_slices_prepare", code, P, P, N.ptr(zero), N.ptr(zero), N.ptr(pins),
           N.ptr(start_d), N.ptr(p2net), None, N.ptr(pins), N.ptr(one), N.ptr(slot_d), N.ptr(prep),
           N.ptr(off), N.ptr(dst), N.ptr(node), N.ptr(meta), st)
    ws = torch.empty(N.query("dp_wa_pins_workspace_bytes", slots, code), dtype=torch.uint8,
                     device=gpu)
    mask, gam = torch.ones(E, dtype=torch.uint8, device=gpu), torch.ones(1, dtype=dtype, device=gpu)
    extent, wl = torch.zeros(E, dtype=dtype, device=gpu), torch.zeros(1, dtype=dtype, device=gpu)
    N.call("dp_wa_forward_slices", code, model, N.ptr(pos), P, P, N.ptr(node), N.ptr(off),
           N.ptr(dst), N.ptr(meta), N.ptr(sl), N.ptr(ln), len(slices), N.ptr(bg), len(big), E,
           None, N.ptr(mask), N.ptr(gam), None, N.ptr(extent), N.ptr(torch.zeros_like(pos)),
           N.ptr(wl), N.ptr(ws), st)
    want = [np.ptp(v[0][~np.isnan(v[0])]) + np.ptp(v[1][~np.isnan(v[1])]) for v in vs]
    assert np.abs(extent.double().cpu().numpy() - want).max() <= 1e-4
