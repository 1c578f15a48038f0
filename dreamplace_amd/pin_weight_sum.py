"""Per-node sum of net weights over the node's pins: drop-in for
dreamplace/ops/pin_weight_sum/pin_weight_sum.py (``PinWeightSum``,
pin_weight_sum.py:30-65); used by the placer's preconditioner."""
import torch
from torch import nn

from . import _native as N
from . import exchange

# Pins from which the sum goes through tiles in LDS (the same bits).  Measured,
# a random load per pin / tiles: FP32 1.8 million pins 11 / 14 us, 3.1 million
# 18 / 17, 9.6 million 111 / 35; FP64 13 / 16, 26 / 21, 146 / 44.
TILE_MIN_PINS = 5 << 19


class PinWeightSum(nn.Module):
    def __init__(self, flat_nodepin=None, nodepin_start=None, pin2net_map=None, num_nodes=None,
                 algorithm='node-by-node'):
        super(PinWeightSum, self).__init__()
        assert flat_nodepin is not None and nodepin_start is not None, \
            "the node-by-node sum needs the node-to-pin CSR (flat_nodepin and nodepin_start)"
        self.flat_nodepin = N.as_i32(flat_nodepin).contiguous()
        self.nodepin_start = N.as_i32(nodepin_start).contiguous()
        self.pin2net_map = N.as_i32(pin2net_map).contiguous()
        self.num_nodes = num_nodes
        self.algorithm = algorithm
        self._plan = N.Derived()
        self._nets()

    def _nets(self):
        """(the net of every node-order pin slot - the two maps in one - or
        None, exchange.weight_tiles of it or None), laid out once, one of the
        two; neither where nothing is kept of the maps (_native.Derived) or
        they hold more than pins; None for maps off the GPU."""
        maps = self.flat_nodepin, self.pin2net_map, self.nodepin_start
        if not all(m.is_cuda for m in maps):
            return None

        def build(pins, nets, start):
            # what lies past the nodes' lists is never read and may name no pin
            if not bool(((pins >= 0) & (pins < nets.numel())).all()):
                return None, None
            slot_net = nets[pins.long()].contiguous()
            x = None
            if pins.numel() >= TILE_MIN_PINS:
                x = exchange.weight_tiles(N.query("dp_wa_tile_pins", N.DP_FLOAT32), slot_net, start)
            return (slot_net, None) if x is None else (None, x)

        return self._plan.get(build, *maps) or (None, None)

    def forward(self, net_weights):
        N.require_gpu(net_weights, name="PinWeightSum")
        w = net_weights.contiguous()
        out = torch.empty(self.num_nodes, dtype=w.dtype, device=w.device)
        plan = self._nets()
        if plan is None:
            raise RuntimeError("PinWeightSum: the maps must be on the GPU")
        nets, x = plan
        code, s = N.dtype_code(w), N.stream_ptr(w.device)
        nphys, n = self.nodepin_start.numel() - 1, int(self.num_nodes)
        if x is not None:
            P = x["cell"].numel()
            ws = torch.empty(P, dtype=w.dtype, device=w.device)
            N.call("dp_pin_weight_sum_tiles", code, N.ptr(w), N.ptr(x["net_tiles"]), x["size"], P,
                   N.ptr(x["cell"]), N.ptr(x["chunk"]), N.ptr(x["delta"]), N.ptr(x["node_tiles"]),
                   len(x["node_tiles"]) - 1, N.ptr(x["node_cell"]), N.ptr(self.nodepin_start),
                   nphys, n, N.ptr(ws), N.ptr(out), s)
        elif nets is not None:
            N.call("dp_pin_weight_sum_slots", code, N.ptr(w), N.ptr(nets),
                   N.ptr(self.nodepin_start), nphys, n, N.ptr(out), s)
        else:
            N.call("dp_pin_weight_sum", code, N.ptr(w), N.ptr(self.flat_nodepin),
                   N.ptr(self.nodepin_start), N.ptr(self.pin2net_map), nphys, n, N.ptr(out), s)
        return out
