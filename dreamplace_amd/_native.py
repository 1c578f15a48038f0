"""ctypes binding of libdreamplace_amd.so (the C ABI declared in
include/dreamplace_amd.h).

PyTorch supplies device memory and the current HIP stream; every call passes
raw pointers.  There is no fallback: if the library is missing, or a tensor
is not on the GPU, the call raises.
"""
import ctypes
import os
import threading

import torch

_HERE = os.path.dirname(os.path.abspath(__file__))
LIB_PATH = os.path.join(_HERE, "libdreamplace_amd.so")

DP_FLOAT32, DP_FLOAT64 = 0, 1
DP_INDEX_INT32, DP_INDEX_INT64 = 0, 1
DP_CONVERT_CPU, DP_CONVERT_GPU = 0, 1
DP_SPECTRAL_FP64, DP_SPECTRAL_FP32, DP_SPECTRAL_BF16X3 = 0, 1, 2
DP_SCATTER_GLOBAL, DP_SCATTER_TILED = 0, 1
DP_LAYOUT_SPLIT, DP_LAYOUT_INTERLEAVED = 0, 1
DP_LAYOUT_FILLERS_FINAL = 0x10
DP_ARITH_BIN_RELATIVE = 0x100
DP_NET_WEIGHTING_ADAMS, DP_NET_WEIGHTING_LILITH = 0, 1
DP_WL_WEIGHTED_AVERAGE, DP_WL_LOGSUMEXP, DP_WL_WEIGHTED_AVERAGE_CENTRED = 0, 1, 2

PRECISIONS = {"fp64": DP_SPECTRAL_FP64, "fp32": DP_SPECTRAL_FP32, "bf16x3": DP_SPECTRAL_BF16X3}

_P = ctypes.c_void_p
_I = ctypes.c_int
_L = ctypes.c_int64
_D = ctypes.c_double
_S = ctypes.c_size_t

# name -> (restype, argtypes)
_SIGNATURES = {
    "dp_last_error": (ctypes.c_char_p, []),
    "dp_version": (_I, []),
    "dp_fixed_point_scale": (_L, [_D, _D, _D, _D]),
    "dp_density_map_workspace_bytes": (_S, [_L, _L, _L, _L, _I, _I]),
    "dp_density_map": (_I, [_I, _P, _L, _P, _P, _P, _P, _P, _P, _D, _D, _D, _D, _D, _D, _L, _L,
                            _I, _I, _I, _I, _L, _P, _P, _P, _P, _P]),
    "dp_density_map_ex": (_I, [_I, _P, _L, _P, _P, _P, _P, _P, _P, _D, _D, _D, _D, _D, _D,
                               _L, _L, _I, _I, _I, _I, _L, _P, _P, _P, _P, _P, _P]),
    "dp_density_map_noalloc": (_I, [_I, _P, _L, _P, _P, _P, _P, _P, _P, _D, _D, _D, _D, _D, _D,
                                    _L, _L, _I, _I, _I, _P, _P, _P, _P]),
    "dp_fixed_density_map": (_I, [_I, _P, _L, _P, _P, _P, _P, _D, _D, _D, _D, _D, _D, _L, _L, _I,
                                  _I, _D, _I, _P, _P, _P]),
    "dp_electric_force": (_I, [_I, _P, _P, _P, _P, _L, _P, _P, _P, _P, _P, _D, _D, _D, _D, _L, _L,
                               _I, _I, _I, _L, _I, _P, _P, _P, _P]),
    "dp_electric_force_fillers_final": (_I, [_I, _P, _P, _P, _P, _L, _P, _P, _P, _P, _P, _D, _D,
                                             _D, _D, _L, _L, _I, _I, _I, _L, _I, _P, _P, _P, _P,
                                             _P, _D, _D, _P]),
    "dp_energy_gradient": (_I, [_I, _P, _P, _P, _L, _P, _P, _P, _P, _P, _D, _D, _D, _D, _L, _L,
                                _I, _I, _I, _P, _P, _P]),
    "dp_reduce_workspace_bytes": (_S, [_L]),
    "dp_density_overflow": (_I, [_I, _P, _L, _D, _P, _P, _P]),
    "dp_spectral_plan_bytes": (_S, [_I, _I, _I]),
    "dp_spectral_plan_init": (_I, [_I, _I, _I, _P, _P]),
    "dp_spectral_workspace_bytes": (_S, [_I, _I, _I]),
    "dp_dct2": (_I, [_I, _P, _I, _I, _P, _P, _P, _P]),
    "dp_idct2": (_I, [_I, _P, _I, _I, _P, _P, _P, _P]),
    "dp_idxst_idct": (_I, [_I, _P, _I, _I, _P, _P, _P, _P]),
    "dp_idct_idxst": (_I, [_I, _P, _I, _I, _P, _P, _P, _P]),
    "dp_poisson_solve": (_I, [_I, _P, _I, _I, _P, _D, _D, _I, _P, _P, _P, _P, _P, _P]),
    "dp_pin_pos_forward": (_I, [_I, _P, _L, _P, _P, _P, _I, _L, _P, _P]),
    "dp_pin_pos_backward": (_I, [_I, _P, _L, _P, _P, _L, _L, _P, _P]),
    "dp_pin_pos_workspace_bytes": (_S, [_I, _L]),
    "dp_pin_pos_forward_tiles": (_I, [_I, _P, _L, _P, _P, _L, _P, _L, _P, _P, _P, _L, _P, _P,
                                      _P, _P]),
    "dp_pin_pos_backward_tiles": (_I, [_I, _P, _L, _L, _P, _P, _P, _P, _L, _P, _P, _L, _L, _P,
                                       _P, _P]),
    "dp_wa_workspace_bytes": (_S, [_L]),
    "dp_wa_merged_forward": (_I, [_I, _P, _L, _P, _P, _L, _P, _P, _P, _P, _P, _P, _P, _P]),
    "dp_lse_merged_forward": (_I, [_I, _P, _L, _P, _P, _L, _P, _P, _P, _P, _P, _P, _P, _P]),
    "dp_wa_merged_backward": (_I, [_I, _P, _P, _L, _P, _P, _P, _P, _P]),
    "dp_wa_merged_backward_recompute": (_I, [_I, _P, _P, _L, _P, _P, _L, _P, _P, _P, _P, _P,
                                             _P]),
    "dp_wa_net_weight_grad": (_I, [_I, _P, _P, _P, _L, _P, _P]),
    "dp_net_weighting": (_I, [_I, _I, _L, _P, _P, _D, _P, _I, _D, _D, _P, _P, _P]),
    "dp_wa_forward_from_nodes": (_I, [_I, _P, _L, _P, _P, _P, _L, _P, _P, _L, _P, _P, _P, _P,
                                      _P, _P, _P, _P]),
    "dp_wa_backward_to_nodes": (_I, [_I, _P, _P, _L, _P, _P, _P, _P, _P, _P, _P, _L, _L, _P, _P]),
    "dp_profile_kernel": (_I, [_I, _P, _P]),
    "dp_wa_pack_nets": (_I, [_P, _L, _P, _P, _P, _P, _P]),
    "dp_wa_prepare_workspace_bytes": (_S, [_L]),
    "dp_wa_pins_prepare": (_I, [_I, _L, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P,
                                _P, _P]),
    "dp_wa_pins_workspace_bytes": (_S, [_L, _I]),
    "dp_wa_forward_pins": (_I, [_I, _P, _L, _L, _P, _P, _P, _P, _P, _L, _P, _L, _L, _P, _P, _P,
                                _P, _P, _P, _P, _P, _P, _P]),
    "dp_wa_forward_pins_centred": (_I, [_I, _P, _L, _L, _P, _P, _P, _P, _P, _L, _P, _L, _L, _P, _P, _P,
                                _P, _P, _P, _P, _P, _P, _P]),
    "dp_lse_forward_pins": (_I, [_I, _P, _L, _L, _P, _P, _P, _P, _P, _L, _P, _L, _L, _P, _P, _P,
                                 _P, _P, _P, _P, _P, _P, _P]),
    "dp_wa_pack_slices": (_I, [_P, _L, _P, _P, _P, _P, _P, _P, _P]),
    "dp_wa_slices_prepare": (_I, [_I, _L, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P,
                                  _P, _P, _P]),
    "dp_wa_forward_slices": (_I, [_I, _I, _P, _L, _L, _P, _P, _P, _P, _P, _P, _L, _P, _L, _L, _P,
                                  _P, _P, _P, _P, _P, _P, _P, _P]),
    "dp_wa_tile_pins": (_I, [_I]),
    "dp_wa_forward_tiles": (_I, [_I, _I, _P, _L, _L, _P, _P, _P, _L, _P, _P, _P, _L, _P, _P,
                                 _P, _P, _P, _P, _L, _P, _L, _L, _P, _P, _P, _P, _P, _P, _P, _P,
                                 _P]),
    "dp_wa_num_partials": (_L, [_L, _L, _L]),
    "dp_node_grad_objective": (_I, [_I, _P, _P, _P, _L, _P, _P, _P, _I, _L, _L, _P, _P, _P, _D,
                                    _D, _P, _P, _P, _P, _P, _L, _P, _P, _D, _P, _P]),
    "dp_wa_pins_slot_weights": (_I, [_I, _L, _P, _P, _P, _P, _P]),
    "dp_node_grad_from_pins": (_I, [_I, _P, _P, _P, _P, _I, _L, _L, _P, _P]),
    "dp_node_grad_preconditioned": (_I, [_I, _P, _P, _P, _P, _I, _L, _L, _P, _P, _P, _D, _D, _P,
                                         _P, _P, _P, _P]),
    "dp_hpwl": (_I, [_I, _P, _L, _P, _P, _L, _P, _P, _P, _P, _P]),
    "dp_step_metrics_workspace_bytes": (_S, []),
    "dp_step_metrics": (_I, [_I, _P, _P, _L, _P, _P, _P, _L, _D, _P, _P, _P]),
    "dp_hpwl_from_nets": (_I, [_I, _P, _P, _L, _P, _P, _P, _P, _P]),
    "dp_move_boundary": (_I, [_I, _P, _L, _P, _P, _D, _D, _D, _D, _L, _L, _P]),
    "dp_filler_tile_keys": (_I, [_I, _P, _L, _L, _D, _D, _D, _D, _I, _I, _D, _D, _P, _P, _P]),
    "dp_permute_fillers_workspace_bytes": (_S, [_I, _L, _I]),
    "dp_permute_fillers": (_I, [_I, _P, _I, _L, _L, _P, _P, _P]),
    "dp_pin_weight_sum_slots": (_I, [_I, _P, _P, _P, _L, _L, _P, _P]),
    "dp_pin_weight_sum_tiles": (_I, [_I, _P, _P, _L, _L, _P, _P, _P, _P, _L, _P, _P, _L, _L, _P,
                                     _P, _P]),
    "dp_pin_weight_sum": (_I, [_I, _P, _P, _P, _P, _L, _L, _P, _P]),
    "dp_optimizer_workspace_bytes": (_S, []),
    "dp_nesterov_extrapolate": (_I, [_I, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P]),
    "dp_nesterov_extrapolate_bounded": (_I, [_I, _L, _P, _P, _P, _P, _P, _P, _P, _P, _P, _P, _D,
                                             _D, _D, _D, _L, _L, _P, _P, _P, _P]),
    "dp_step_norms": (_I, [_I, _L, _P, _P, _P, _P, _P, _P, _P]),
    "dp_l1_norm": (_I, [_I, _L, _P, _P, _P, _P]),
    "dp_precondition": (_I, [_I, _P, _L, _P, _P, _P, _D, _P]),
    # host-only Bookshelf reader
    "dp_bookshelf_read": (_I, [ctypes.c_char_p, _I, ctypes.POINTER(_P)]),
    "dp_bookshelf_sizes": (_I, [_P, _P]),
    "dp_bookshelf_export": (_I, [_P] + [_P] * 21),
    "dp_bookshelf_free": (None, [_P]),
    "dp_rect_union_area": (_D, [_L, _P, _P, _P, _P, _P]),
}

_lib = None
_lock = threading.Lock()


def lib():
    """The loaded native library; raises RuntimeError if it is not built."""
    global _lib
    if _lib is None:
        with _lock:
            if _lib is None:
                if not os.path.exists(LIB_PATH):
                    raise RuntimeError(
                        "dreamplace_amd: native library %s is not built; run "
                        "`python -m dreamplace_amd.build` (hipcc, gfx950)" % LIB_PATH)
                L = ctypes.CDLL(LIB_PATH)
                for name, (res, args) in _SIGNATURES.items():
                    fn = getattr(L, name)
                    fn.restype = res
                    fn.argtypes = args
                _lib = L
    return _lib


def exported_symbols():
    return list(_SIGNATURES)


def call(name, *args):
    """Call a status-returning entry point and raise on a non-zero status."""
    rc = getattr(_lib or lib(), name)(*args)
    if rc != 0:
        msg = lib().dp_last_error().decode(errors="replace")
        raise RuntimeError("%s failed (status %d): %s" % (name, rc, msg))


def query(name, *args):
    return getattr(_lib or lib(), name)(*args)


def ptr(t):
    """Device pointer of a tensor (None for None), as the integer that a
    void* argument takes."""
    return None if t is None else t.data_ptr()


def ptr_np(a):
    """Host pointer of a C-contiguous numpy array (None for None)."""
    if a is None:
        return None
    if not a.flags["C_CONTIGUOUS"]:
        raise ValueError("host array must be C-contiguous")
    return ctypes.c_void_p(a.ctypes.data)


def host_doubles(values):
    """A host double array for an argument read during the call (None for None)."""
    if values is None:
        return None
    return (ctypes.c_double * len(values))(*[float(v) for v in values])


def require_gpu(*tensors, name="dreamplace_amd"):
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("%s: tensors must be on the GPU (got a %s tensor); the "
                               "dreamplace_amd ops run only on the HIP path" % (name, t.device))


def require_contiguous(*tensors, name="dreamplace_amd"):
    for t in tensors:
        if t is not None and not t.is_contiguous():
            raise RuntimeError("%s: tensor must be contiguous" % name)


def dtype_code(t):
    if t.dtype == torch.float32:
        return DP_FLOAT32
    if t.dtype == torch.float64:
        return DP_FLOAT64
    raise RuntimeError("dreamplace_amd: dtype %s not implemented (float32/float64 only)" % t.dtype)


_raw_stream = getattr(torch._C, "_cuda_getCurrentRawStream", None)


def stream_ptr(device=None):
    """The current stream's handle on a device (default: the current one)."""
    index = getattr(device, "index", None)
    if _raw_stream is not None and index is not None:
        return _raw_stream(index)
    return torch.cuda.current_stream(device).cuda_stream


def as_i32(t):
    return t if t.dtype == torch.int32 else t.to(torch.int32)


def as_u8(t):
    """A mask as bytes of 0 and 1, a bool tensor's in a copy: what becomes of it
    between a forward and its backward stays out of the latter."""
    if t is None or t.dtype == torch.uint8:
        return t
    if t.dtype == torch.bool:  # a conversion takes 14.6 us for 9.6 million, this copy 5.2
        return t.view(torch.uint8).clone(memory_format=torch.contiguous_format)
    return t.to(torch.uint8)


class Derived:
    """Tensors computed once from static index maps and kept while they are
    the same objects, unmodified and at the same addresses: get(build, *maps).
    It holds the maps, so none can be replaced by another, and rebuilds after
    an in-place change (one that torch does not count, through .data or a raw
    pointer, is not seen).  A build is waited for, so that any stream may use
    it, and what another one uses is freed only after it.  A copy or a saved
    one holds nothing.
    get is None where nothing may be kept, and the caller works on the maps
    themselves: of inference tensors, whose changes are not counted, and while
    a graph is captured, which would only record a build and would hold the
    addresses of what a later change of the maps frees."""

    def __init__(self):
        # maps, their versions and addresses, the value, the stream that built it
        self._state = (None, None, None, None)

    def __reduce__(self):
        return Derived, ()  # a copied map's versions start anew

    def get(self, build, *maps):
        if any(m.is_inference() for m in maps) or torch.cuda.is_current_stream_capturing():
            return None
        key = tuple((m._version, m.data_ptr()) for m in maps)
        stream = stream_ptr(maps[0].device)
        held, seen, value, built = self._state
        if held is None or any(a is not b for a, b in zip(held, maps)) or seen != key:
            value, built = build(*maps), stream
            torch.cuda.current_stream(maps[0].device).synchronize()
            self._state = (maps, key, value, built)
        if stream != built:
            for t in _tensors(value):
                t.record_stream(torch.cuda.current_stream(maps[0].device))
        return value


def _tensors(value):
    """The tensors in a nest of tuples and dicts."""
    if torch.is_tensor(value):
        yield value
    elif isinstance(value, (tuple, dict)):
        for v in value.values() if isinstance(value, dict) else value:
            yield from _tensors(v)


class Workspace:
    """Grow-only scratch buffers, one per (key, device)."""

    def __init__(self):
        self._bufs = {}

    def get(self, key, nbytes, device):
        k = (key, str(device))
        b = self._bufs.get(k)
        if b is None or b.numel() < nbytes:
            b = torch.empty(max(int(nbytes), 256), dtype=torch.uint8, device=device)
            self._bufs[k] = b
        return b


workspace = Workspace()
