"""What the ops keep of static index maps: nothing while a graph is captured or
of inference tensors, and nothing that outlives a change or goes with a copy."""
import copy
import pickle

import pytest
import torch

from dreamplace_amd import _native as N


class Stream:
    """A stream on the CPU."""
    cuda_stream = 0

    def __init__(self, *a):
        pass

    def synchronize(self):
        pass


@pytest.fixture
def cpu_stream(monkeypatch):
    monkeypatch.setattr(torch.cuda, "current_stream", Stream)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)


def sums():
    """A Derived, its map and the call that keeps the map's sum."""
    d, m = N.Derived(), torch.arange(5)
    return d, m, lambda d, m: d.get(lambda x: (x.sum(),), m)


def test_kept(cpu_stream):
    d, m, get = sums()
    first = get(d, m)
    assert get(d, m) is first and int(first[0]) == 10
    m[0] = 4
    assert int(get(d, m)[0]) == 14 and int(get(d, m.clone())[0]) == 14


@pytest.mark.parametrize("copy_of", [copy.deepcopy, lambda x: pickle.loads(pickle.dumps(x))],
                         ids=["copied", "saved"])
def test_copies(cpu_stream, copy_of):
    """A copy after a change: the copied map counts its own changes anew, and
    may come to the count that the plan was made at."""
    d, m, get = sums()
    first = copy_of(m)._version
    while m._version < first:
        m[0] = 0
    get(d, m)
    m[0] = 4
    d, m = copy_of((d, m))
    assert int(get(d, m)[0]) == 14


def test_other_storage(cpu_stream):
    d, m, get = sums()
    get(d, m)
    m.data = torch.arange(7)
    assert int(get(d, m)[0]) == 21


def test_nothing_kept(cpu_stream, monkeypatch):
    d, m, get = sums()
    with torch.inference_mode():
        assert get(d, torch.arange(5)) is None
    get(d, m)
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: True)
    assert get(d, m) is None
    m[0] = 4
    assert get(d, m) is None
    monkeypatch.setattr(torch.cuda, "is_current_stream_capturing", lambda: False)
    assert int(get(d, m)[0]) == 14


def netlist(gpu, pins, nphys, nets):
    """(pin2node, node order of the pins, its start array, pin2net)"""
    g = torch.Generator(device=gpu).manual_seed(6)
    p2n = torch.randint(0, nphys, (pins,), generator=g, device=gpu)
    order = torch.sort(p2n, stable=True).indices.int()
    start = torch.zeros(nphys + 1, dtype=torch.int32, device=gpu)
    start[1:] = torch.bincount(p2n, minlength=nphys).cumsum(0)
    return p2n, order, start, torch.randint(0, nets, (pins,), generator=g, device=gpu).int()


@pytest.mark.gpu
@pytest.mark.parametrize("least", [1, 1 << 40], ids=["tiles", "few"])
def test_capture(gpu, monkeypatch, least):
    """Maps changed in place before a capture, then eager calls before the first
    replay, then maps changed between replays: every result is the maps'."""
    from dreamplace_amd import pin_pos, pin_weight_sum
    print("case capture of kept plans %d" % least, flush=True)
    monkeypatch.setattr(pin_pos, "TILE_MIN_PINS", least)
    monkeypatch.setattr(pin_weight_sum, "TILE_MIN_PINS", least)
    pins, nphys, nets = 5000, 700, 900
    p2n, order, start, p2e = netlist(gpu, pins, nphys, nets)
    off, pos = torch.rand(pins, device=gpu), torch.rand(2 * nphys, device=gpu)
    w = torch.rand(nets, device=gpu, dtype=torch.float64)
    a = pin_pos.PinPos(off, off, p2n, order, start, nphys)
    b = pin_weight_sum.PinWeightSum(order, start, p2e, nphys)

    def other_maps():  # the same numbers of pins, other pins and other nets
        a.pin2node_map.copy_(a.pin2node_map.flip(0))
        order.copy_(torch.sort(a.pin2node_map, stable=True).indices)
        p2e.copy_(p2e.flip(0))

    def check(out, sums):
        torch.cuda.synchronize()
        n = a.pin2node_map
        assert torch.equal(out, torch.cat([off + pos[:nphys][n], off + pos[nphys:][n]]))
        ref = torch.zeros(nphys, dtype=w.dtype, device=gpu).index_add_(0, n, w[p2e.long()])
        assert (sums - ref).abs().max() <= 1e-13 * ref.max()

    check(a(pos), b(w))
    other_maps()
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out, sums = a(pos), b(w)
    check(a(pos), b(w))  # eager, with nothing replayed yet
    for _ in range(3):
        out.zero_(), sums.zero_()
        graph.replay()
        check(out, sums)
        other_maps()
        check(a(pos), b(w))


@pytest.mark.gpu
@pytest.mark.parametrize("least", [1, 1 << 40], ids=["tiles", "few"])
@pytest.mark.parametrize("past", [-1, 1 << 30])
def test_padded_map(gpu, monkeypatch, past, least):
    """A node-to-pin map longer than its start array says, the rest no pin."""
    from dreamplace_amd import pin_weight_sum
    print("case padded map %d %d" % (past, least), flush=True)
    monkeypatch.setattr(pin_weight_sum, "TILE_MIN_PINS", least)
    p2n, order, start, p2e = netlist(gpu, 5000, 700, 900)
    w = torch.rand(900, device=gpu)
    want = pin_weight_sum.PinWeightSum(order, start, p2e, 800)(w)
    padded = torch.cat([order, order.new_full((100,), past)])
    assert torch.equal(pin_weight_sum.PinWeightSum(padded, start, p2e, 800)(w), want)


def test_few_positions(monkeypatch):
    """Positions of fewer nodes than the physical ones, the last of which have no
    pins: no node tile, which reads all of them."""
    from dreamplace_amd import pin_pos
    p2n = torch.arange(12) % 3
    start = torch.tensor([0, 4, 8, 12, 12, 12])
    op = pin_pos.PinPos(torch.rand(12), torch.rand(12), p2n, p2n.argsort(stable=True), start, 5)
    monkeypatch.setattr(op, "_plan", lambda dtype: "tiles")
    taken = []
    monkeypatch.setattr(pin_pos.PinPosFunction, "apply", lambda *a: taken.append(a[-1]))
    for nodes in (3, 4, 5, 6):
        op(torch.rand(2 * nodes))
    assert taken == [None, None, "tiles", "tiles"]


@pytest.mark.gpu
@pytest.mark.parametrize("least", [1, 1 << 40], ids=["tiles", "few"])
def test_other_stream(gpu, monkeypatch, least):
    """Modules that are dropped while another stream has yet to run their call:
    what it reads is not given to a new tensor before it has."""
    from dreamplace_amd import pin_pos, pin_weight_sum
    print("case kept plans on another stream %d" % least, flush=True)
    monkeypatch.setattr(pin_pos, "TILE_MIN_PINS", least)
    monkeypatch.setattr(pin_weight_sum, "TILE_MIN_PINS", least)
    pins, nphys, nets = 50000, 7000, 9000
    p2n, order, start, p2e = netlist(gpu, pins, nphys, nets)
    off, pos = torch.rand(pins, device=gpu), torch.rand(2 * nphys, device=gpu)
    w = torch.rand(nets, device=gpu)
    a = pin_pos.PinPos(off, off, p2n, order, start, nphys)
    b = pin_weight_sum.PinWeightSum(order, start, p2e, nphys)
    want = a(pos).clone(), b(w).clone()
    kept = [t for d in (a._tiles, b._plan) for t in N._tensors(d._state[2])]
    held = {t.data_ptr(): t.numel() * t.element_size() for t in kept}
    assert (len(held) > 8) == (least == 1) and held
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        torch.cuda._sleep(200000000)
        got = a(pos), b(w)
        done = torch.cuda.Event()
        done.record()
    del a, b, kept
    new = [torch.zeros(n, dtype=torch.uint8, device=gpu) for n in held.values()]
    if not done.query():  # else the memory was free to give
        assert not held.keys() & {t.data_ptr() for t in new}
    torch.cuda.synchronize()
    assert torch.equal(got[0], want[0]) and torch.equal(got[1], want[1])
