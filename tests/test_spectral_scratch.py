"""A grid's plan is shared by all callers: each call has scratch that no other
call in flight writes, on another stream, in another thread or in a graph; and
a plan first asked for while a graph is captured is the graph's own."""
import pytest
import torch

from dreamplace_amd import _native as N
from dreamplace_amd import spectral


@pytest.fixture
def calls(monkeypatch):
    """Calls of the library on CPU tensors, recorded: (name, scratch, stream);
    `.stream` is the current one, `.during` runs within the next call."""
    class Calls(list):
        stream, during, capturing = 1, None, False

        def __call__(self, name, *args):
            if name.endswith("_init"):
                return
            self.append((name, args[-2], args[-1]))
            during, self.during = self.during, None
            if during:
                during()

    calls = Calls()
    monkeypatch.setattr(N, "call", calls)
    monkeypatch.setattr(N, "stream_ptr", lambda device=None: calls.stream)
    monkeypatch.setattr(N, "require_gpu", lambda *a, **k: None)
    monkeypatch.setattr(spectral, "capturing", lambda: calls.capturing)
    monkeypatch.setattr(spectral, "_plans", {})
    return calls


def test_scratch(calls):
    plan = spectral.get_plan(32, 64, "fp32", "cpu")
    x = torch.zeros(32, 64)
    plan.dct2(x)
    plan.poisson(x, 1.0, 1.0)
    assert calls[0][1] == calls[1][1]          # one stream: the calls are in order
    calls.stream = 2
    calls.during = lambda: (setattr(calls, "stream", 1), plan.idct2(x))
    plan.dct2(x)
    assert calls[2][1] != calls[3][1] == calls[0][1]
    calls.during = lambda: plan.idct2(x)       # another thread, the same stream
    plan.dct2(x)
    assert calls[4][2] == calls[5][2] and calls[4][1] != calls[5][1]
    for calls.stream in range(10, 30):
        plan.dct2(x)
    assert len(plan._free) <= spectral.MAX_FREE
    assert {c[2] for c in calls} == {1, 2, *range(10, 30)}


def test_capture(calls):
    plan = spectral.get_plan(32, 64, "fp32", "cpu")
    x = torch.zeros(32, 64)
    plan.dct2(x)
    kept = dict(plan._free)
    calls.capturing = plan.gpu = True
    plan.dct2(x)
    assert calls[1][1] != calls[0][1] and plan._free == kept
    assert spectral.get_plan(32, 64, "fp32", "cpu") is plan


@pytest.mark.gpu
def test_replays(gpu):
    """A captured solve, replayed on one stream beside eager ones on another."""
    print("case captured solve", flush=True)
    g = torch.Generator(device=gpu).manual_seed(3)
    maps = torch.rand(2, 512, 512, generator=g, device=gpu)
    plan = spectral.get_plan(512, 512, "fp32", gpu)
    want = [plan.poisson(m, 1.0, 1.0) for m in maps]
    torch.cuda.synchronize()
    graph, side = torch.cuda.CUDAGraph(), torch.cuda.Stream()
    with torch.cuda.graph(graph):
        got = plan.poisson(maps[0], 1.0, 1.0)
    for _ in range(5):
        for t in got:
            t.zero_()
        torch.cuda.synchronize()
        with torch.cuda.stream(side):
            eager = [plan.poisson(maps[1], 1.0, 1.0) for _ in range(8)]
        for _ in range(8):
            graph.replay()
        torch.cuda.synchronize()
        for res, ref in [(got, want[0])] + [(e, want[1]) for e in eager]:
            assert all(torch.equal(a, b) for a, b in zip(res, ref))


@pytest.mark.gpu
@pytest.mark.parametrize("shape", [(64, 256), (72, 56)], ids=str)
def test_plan_in_capture(gpu, monkeypatch, shape):
    """A grid first asked for during a capture: an eager call before the first
    replay has tables of its own."""
    print("case plan in capture %s" % (shape,), flush=True)
    monkeypatch.setattr(spectral, "_plans", {})
    x = torch.rand(*shape, generator=torch.Generator(device=gpu).manual_seed(4), device=gpu)
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = spectral.get_plan(*shape, "fp32", gpu).dct2(x)
    want = spectral.get_plan(*shape, "fp32", gpu).dct2(x)
    torch.cuda.synchronize()
    assert float(want[0, 0]) == pytest.approx(4 * float(x.mean()), rel=1e-5)
    for _ in range(3):
        got.zero_()
        graph.replay()
        assert torch.equal(got, want)
        assert torch.equal(spectral.get_plan(*shape, "fp32", gpu).dct2(x), want)
