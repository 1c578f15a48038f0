"""Pin positions from cell positions: drop-in for
dreamplace/ops/pin_pos/pin_pos.py (``PinPos``, pin_pos.py:103-156).

Forward: pin_pos[p] = offset[p] + pos[pin2node[p]] (x block then y block).
Backward: node gradient = sum of pin gradients over the node's CSR pins
(flat_node2pin_map / flat_node2pin_start_map); fillers receive 0.
Both algorithm names ('segment', 'node-by-node') run the same kernels.
"""
import torch
from torch import nn
from torch.autograd import Function

from . import _native as N
from . import exchange

# Pins from which the module permutes between node and pin order through tiles
# in LDS (the same bits as the plain kernels).  Measured, plain / tiles, forward
# and backward: FP32 1.1 million pins 13 / 20 us and 38 / 50 (host-bound), 1.8
# million 21 / 20 and 53 / 31, 4.4 million 93 / 29 and 153 / 27, 10.9 million
# 331 / 100 and 428 / 83; FP64 1.1 million 19 / 20 and 36 / 32, 4.4 million
# 139 / 59 and 172 / 58, 10.9 million 413 / 184 and 444 / 140.
TILE_MIN_PINS = 3 << 19


class PinPosFunction(Function):
    @staticmethod
    def forward(ctx, pos, pin_offset_x, pin_offset_y, pin2node_map, flat_node2pin_map,
                flat_node2pin_start_map, num_physical_nodes, tiles=None):
        """tiles (optional): exchange.pin_tiles of the maps, for pos.dtype."""
        N.require_gpu(pos, pin_offset_x, pin2node_map, name="PinPos")
        pos = pos.view(pos.numel()).contiguous()
        num_nodes = pos.numel() // 2
        num_pins = pin2node_map.numel()
        out = torch.empty(2 * num_pins, dtype=pos.dtype, device=pos.device)
        if tiles is not None:
            code = N.dtype_code(pos)
            ws = torch.empty(N.query("dp_pin_pos_workspace_bytes", code, num_pins),
                             dtype=torch.uint8, device=pos.device)
            N.call("dp_pin_pos_forward_tiles", code, N.ptr(pos), num_nodes, N.ptr(pin_offset_x),
                   N.ptr(pin_offset_y), num_pins, N.ptr(tiles["node_tiles"]),
                   len(tiles["node_tiles"]) - 1, N.ptr(tiles["place_node"]),
                   N.ptr(tiles["node_chunk"]), N.ptr(tiles["node_delta"]), tiles["size"], N.ptr(tiles["cell"]), N.ptr(ws),
                   N.ptr(out), N.stream_ptr(pos.device))
        else:
            idx_type = N.DP_INDEX_INT64 if pin2node_map.dtype == torch.int64 else N.DP_INDEX_INT32
            p2n = (pin2node_map if pin2node_map.dtype in (torch.int32, torch.int64)
                   else pin2node_map.long())
            N.call("dp_pin_pos_forward", N.dtype_code(pos), N.ptr(pos), num_nodes,
                   N.ptr(pin_offset_x), N.ptr(pin_offset_y), N.ptr(p2n.contiguous()), idx_type,
                   num_pins, N.ptr(out), N.stream_ptr(pos.device))
        ctx.num_nodes = num_nodes
        ctx.num_pins = num_pins
        ctx.num_physical_nodes = int(num_physical_nodes)
        ctx.flat_node2pin_map = N.as_i32(flat_node2pin_map).contiguous()
        ctx.flat_node2pin_start_map = N.as_i32(flat_node2pin_start_map).contiguous()
        ctx.tiles = tiles
        return out

    @staticmethod
    def backward(ctx, grad_pin_pos):
        g = grad_pin_pos.contiguous()
        out = torch.empty(2 * ctx.num_nodes, dtype=g.dtype, device=g.device)
        x = ctx.tiles
        if x is not None:
            code = N.dtype_code(g)
            ws = torch.empty(N.query("dp_pin_pos_workspace_bytes", code, ctx.num_pins),
                             dtype=torch.uint8, device=g.device)
            N.call("dp_pin_pos_backward_tiles", code, N.ptr(g), ctx.num_pins, x["size"],
                   N.ptr(x["cell"]), N.ptr(x["chunk"]), N.ptr(x["delta"]), N.ptr(x["node_tiles"]),
                   len(x["node_tiles"]) - 1, N.ptr(x["node_cell"]),
                   N.ptr(ctx.flat_node2pin_start_map), ctx.num_physical_nodes, ctx.num_nodes,
                   N.ptr(ws), N.ptr(out), N.stream_ptr(g.device))
        else:
            N.call("dp_pin_pos_backward", N.dtype_code(g), N.ptr(g), ctx.num_pins,
                   N.ptr(ctx.flat_node2pin_map), N.ptr(ctx.flat_node2pin_start_map),
                   ctx.num_physical_nodes, ctx.num_nodes, N.ptr(out), N.stream_ptr(g.device))
        return (out,) + (None,) * 7


class PinPos(nn.Module):
    def __init__(self, pin_offset_x, pin_offset_y, pin2node_map, flat_node2pin_map,
                 flat_node2pin_start_map, num_physical_nodes, algorithm='segment'):
        super(PinPos, self).__init__()
        self.pin_offset_x = pin_offset_x
        self.pin_offset_y = pin_offset_y
        self.pin2node_map = pin2node_map.long()
        self.flat_node2pin_map = flat_node2pin_map
        self.flat_node2pin_start_map = flat_node2pin_start_map
        self.num_physical_nodes = num_physical_nodes
        self.algorithm = algorithm
        self._tiles = N.Derived()
        self._plan(pin_offset_x.dtype)

    def _plan(self, dtype):
        """exchange.pin_tiles of the maps, or None where the plain kernels are
        taken: few pins, maps that the tiles do not apply to, or where no plan
        is kept (_native.Derived)."""
        maps = self.pin2node_map, self.flat_node2pin_map, self.flat_node2pin_start_map
        if maps[0].numel() < TILE_MIN_PINS or not all(m.is_cuda for m in maps):
            return None
        cap = N.query("dp_wa_tile_pins", N.DP_FLOAT64 if dtype == torch.float64 else N.DP_FLOAT32)
        sizes = cap, int(self.num_physical_nodes)
        kept = self._tiles.get(lambda *m: (sizes, exchange.pin_tiles(cap, *m, sizes[1])), *maps)
        return kept[1] if kept is not None and kept[0] == sizes else None

    def forward(self, pos):
        assert pos.numel() % 2 == 0
        # the node tiles hold every physical node, with or without pins
        whole = pos.numel() >= 2 * int(self.num_physical_nodes)
        return PinPosFunction.apply(pos, self.pin_offset_x, self.pin_offset_y, self.pin2node_map,
                                    self.flat_node2pin_map, self.flat_node2pin_start_map,
                                    self.num_physical_nodes,
                                    self._plan(pos.dtype) if whole else None)
