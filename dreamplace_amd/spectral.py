"""Spectral transforms and the Poisson solve: fast transforms on grids whose
sides are powers of two from 32 to 4096, dense products on the matrix cores on
any other.

``SpectralPlan`` holds the twiddle tables or the cosine / sine matrices of an
M x N grid for one arithmetic form ("fp64", "fp32" or "bf16x3"; the fast
transforms of the last are FP32 throughout) and scratch for the transforms;
it wraps dp_dct2 / dp_idct2 / dp_idxst_idct / dp_idct_idxst and
dp_poisson_solve of libdreamplace_amd.  get_plan shares one plan per grid, form
and device among all modules, threads and streams.
"""
import torch

from . import _native as N


def default_precision(dtype):
    return "fp64" if dtype == torch.float64 else "fp32"


def data_dtype(precision):
    return torch.float64 if precision == "fp64" else torch.float32


_is_capturing = getattr(torch._C, "_cuda_isCurrentStreamCapturing", None)


def capturing():
    """Whether a graph is being captured on the current stream."""
    return _is_capturing is not None and _is_capturing()


MAX_FREE = 4  # streams whose scratch a plan keeps (2048 x 2048 in FP32: 118 MB each)


class SpectralPlan:
    def __init__(self, M, N_, precision, device):
        if precision not in N.PRECISIONS:
            raise ValueError("precision must be one of %s" % sorted(N.PRECISIONS))
        self.M, self.N = int(M), int(N_)
        self.precision = precision
        self.code = N.PRECISIONS[precision]
        self.device = torch.device(device)
        self.dtype = data_dtype(precision)
        nbytes = N.query("dp_spectral_plan_bytes", self.M, self.N, self.code)
        self.plan = torch.empty(nbytes, dtype=torch.uint8, device=self.device)
        self._tables = N.ptr(self.plan)
        N.call("dp_spectral_plan_init", self.M, self.N, self.code, self._tables,
               N.stream_ptr(self.device))
        self.gpu = self.device.type == "cuda"
        if self.gpu and not capturing():
            # the tables, for whichever stream reads them first
            torch.cuda.current_stream(self.device).synchronize()
        self._ws_bytes = N.query("dp_spectral_workspace_bytes", self.M, self.N, self.code)
        self._free = {}  # a stream's handle -> the scratch that its last call has left

    def scratch(self):
        """Scratch for a caller whose calls are in order to keep (poisson's ws)."""
        return torch.empty(self._ws_bytes, dtype=torch.uint8, device=self.device)

    def _take(self, stream):
        """(scratch, its address, whether to keep it) for one call on `stream`, to
        be given back (_give) once that is queued: what the last call on the same
        stream has left, which the stream orders before this one; new memory where
        another thread's call has it, or under capture, as a graph's replays keep
        no order with the calls outside.  At most MAX_FREE streams' scratch is
        kept."""
        graph = self.gpu and capturing()
        held = None if graph else self._free.pop(stream, None)
        if held is None:
            ws = self.scratch()
            held = ws, ws.data_ptr(), not graph
        return held

    def _give(self, stream, held):
        if held[2] and len(self._free) < MAX_FREE:
            self._free[stream] = held

    def _check(self, x):
        if not x.is_cuda:
            N.require_gpu(x, name="SpectralPlan")
        if x.dtype != self.dtype:
            raise RuntimeError("SpectralPlan(%s) expects %s data, got %s" % (self.precision, self.dtype, x.dtype))
        if x.shape[-2:] != (self.M, self.N):
            raise RuntimeError("SpectralPlan is for %dx%d grids, got %s" % (self.M, self.N, tuple(x.shape)))
        return x.contiguous()

    def transform(self, name, x, out=None):
        x = self._check(x)
        if out is None:
            out = torch.empty(self.M, self.N, dtype=self.dtype, device=self.device)
        stream = N.stream_ptr(self.device)
        held = self._take(stream)
        N.call(name, self.code, self._tables, self.M, self.N, N.ptr(x), N.ptr(out), held[1], stream)
        self._give(stream, held)
        return out

    def dct2(self, x, out=None):
        return self.transform("dp_dct2", x, out)

    def idct2(self, x, out=None):
        return self.transform("dp_idct2", x, out)

    def idxst_idct(self, x, out=None):
        return self.transform("dp_idxst_idct", x, out)

    def idct_idxst(self, x, out=None):
        return self.transform("dp_idct_idxst", x, out)

    def poisson(self, density_map, bin_size_x, bin_size_y, compute_potential=True,
                compute_energy=True, out=None, ws=None):
        """(field_x, field_y, potential or None, energy 0-dim tensor or None).
        With out and ws (scratch()) a call allocates nothing."""
        d = self._check(density_map)
        if out is None:
            fx = torch.empty(self.M, self.N, dtype=self.dtype, device=self.device)
            fy = torch.empty_like(fx)
            phi = torch.empty_like(fx) if compute_potential else None
            energy = torch.empty((), dtype=self.dtype, device=self.device) if compute_energy else None
        else:
            fx, fy, phi, energy = out
        stream = N.stream_ptr(self.device)
        held = self._take(stream) if ws is None else (ws, ws.data_ptr(), False)
        N.call("dp_poisson_solve", self.code, self._tables, self.M, self.N, N.ptr(d),
               float(bin_size_x), float(bin_size_y), 1 if compute_potential else 0, N.ptr(fx),
               N.ptr(fy), N.ptr(phi), N.ptr(energy), held[1], stream)
        self._give(stream, held)
        return fx, fy, phi, energy


_plans = {}


def get_plan(M, N_, precision, device):
    key = (int(M), int(N_), precision, torch.device(device))
    p = _plans.get(key)
    if p is None:
        p = SpectralPlan(M, N_, precision, device)
        # while a graph is captured the tables are only recorded: the graph's own
        if not (p.gpu and capturing()):
            _plans[key] = p
    return p
