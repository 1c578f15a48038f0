"""One evaluation of the global-placement objective and its gradient.

``PlacementObjective.evaluate(pos)`` computes

    obj  = WA(pin_pos(pos)) + density_weight * E(pos)
    grad = d obj / d pos

exactly as ``PlaceObj.obj_and_grad_fn`` does (dreamplace/PlaceObj.py:394-411,
without the preconditioner), on preallocated device buffers and with no
autograd graph or host synchronisation.  Three schedules:

* ``schedule="pins"``: the WA forward carries pin positions to net order (a few
  lanes per net, nets sorted by degree) and writes each pin's weighted
  derivative in node order, so the backward is a contiguous per-node sum
  (dp_wa_forward_slices / dp_node_grad_from_pins; for a large netlist both
  permutations go through tiles in LDS, dp_wa_forward_tiles);
* ``fused=True``: pin positions are formed inside the WA kernel, and the WA
  backward, the pin-to-node sum and the gradient combine are one node-parallel
  pass (dp_wa_forward_from_nodes / dp_wa_backward_to_nodes);
* ``fused=False``: the reference's op sequence, one C-ABI call per op
  (pin_pos, WA forward, density, solve, force, WA backward, pin_pos backward,
  add).

Both give the same objective and gradient (the fused kernels keep the
per-element arithmetic and summation order).
"""
import ctypes

import numpy as np
import torch

from . import _native as N
from . import exchange
from .electric_overflow import MAX_TILES
from .electric_potential import ElectricPotential


def pack_slices(netpin_start):
    """dp_wa_pack_slices on a host CSR start array: (slices [ns, 2], lane_nets
    [64 ns, 2], big [nb, 4], net_slot [E], num_slots), net_slot[e] the slot of
    net e's first pin (slice_slots: of every pin)."""
    start = np.ascontiguousarray(netpin_start, dtype=np.int32)
    E = len(start) - 1
    cap = (E + int(start[-1]) // 2) // 64 + 6
    slices = np.zeros(2 * cap, dtype=np.int32)
    lanes = np.zeros(128 * cap, dtype=np.int32)
    big = np.zeros(4 * max(E, 1), dtype=np.int32)
    net_slot = np.zeros(max(E, 1), dtype=np.int32)
    ns, nb, slots = ctypes.c_int64(0), ctypes.c_int64(0), ctypes.c_int64(0)
    vp = lambda a: a.ctypes.data_as(ctypes.c_void_p)
    N.call("dp_wa_pack_slices", vp(start), E, vp(slices), ctypes.byref(ns), vp(lanes), vp(big),
           ctypes.byref(nb), vp(net_slot), ctypes.byref(slots))
    return (slices[:2 * ns.value].reshape(-1, 2), lanes[:128 * ns.value].reshape(-1, 2),
            big[:4 * nb.value].reshape(-1, 4), net_slot[:E], slots.value)


def slice_slots(first, rank, degree):
    """The slots of pins `rank` of nets of `degree` pins whose first pin has
    slot `first`, in dp_wa_pack_slices' layout (tensors or arrays)."""
    lanes = 1 + (degree > 4) * 1 + (degree > 8) * 2 + (degree > 16) * 4 + (degree > 32) * 8
    lanes = lanes * (degree <= 64) + 64 * (degree > 64)
    return first + 64 * (rank // lanes) + rank % lanes


def movable_netlist_order(dd):
    """An order of the movable cells for DeviceDesign.reorder_movables: by
    the first slot, in the wirelength pass's slice order (dp_wa_pack_slices),
    among each cell's pins; cells without pins last, in their order.  The
    pass's two permutations (node order <-> slice order) are cut into tiles
    or, on small netlists, scattered 8-byte stores; both run over longer
    stretches when neighbouring cells' pins are near each other, and in this
    order each cell's first pin lands next to its neighbours'."""
    dev = dd.device
    st = dd.flat_net2pin_start_map.long()
    E, P = st.numel() - 1, dd.num_pins
    _, _, _, net_slot, slots = pack_slices(st.cpu().numpy())
    lens = st[1:] - st[:-1]
    net_of_flat = torch.repeat_interleave(torch.arange(E, device=dev), lens)
    rank = torch.arange(P, device=dev) - st[net_of_flat]
    slot = slice_slots(torch.from_numpy(net_slot.astype(np.int64)).to(dev)[net_of_flat], rank,
                       lens[net_of_flat])
    node = dd.pin2node_map.long()[dd.flat_net2pin_map.long()]
    first = torch.full((dd.num_nodes,), slots, dtype=torch.int64, device=dev)
    first.scatter_reduce_(0, node, slot, "amin")
    return torch.argsort(first[:dd.num_movable_nodes], stable=True)


class DeviceDesign:
    """The arrays of a design (a dict such as dreamplace_amd.synth.make_design
    returns) as device tensors with the index types the kernels take."""

    INT_KEYS = ("pin2node_map", "pin2net_map", "flat_net2pin_map", "flat_net2pin_start_map",
                "flat_node2pin_map", "flat_node2pin_start_map", "sorted_node_map")
    U8_KEYS = ("net_mask_all", "net_mask_ignore_large_degrees", "pin_mask_ignore_fixed_macros")

    def __init__(self, d, device, dtype=None):
        self.scalars = {k: v for k, v in d.items() if not isinstance(v, np.ndarray)}
        dt = dtype if dtype is not None else torch.from_numpy(d["pos"][:1]).dtype
        self.dtype = dt
        self.device = torch.device(device)
        self.t = {}
        for k, v in d.items():
            if not isinstance(v, np.ndarray):
                continue
            x = torch.from_numpy(np.ascontiguousarray(v))
            if k in self.INT_KEYS:
                x = x.to(torch.int32)
            elif k in self.U8_KEYS:
                x = x.to(torch.uint8)
            elif k == "movable_macro_mask":
                x = x.to(torch.bool)
            elif x.is_floating_point():
                x = x.to(dt)
            self.t[k] = x.to(self.device, copy=True)  # never aliases the caller's arrays

    def uniform_fillers(self):
        """Whether every filler has the same size (PlaceDB.py:917-936 makes
        them so); only then may their order change."""
        n, nf = self.num_nodes, self.num_filler_nodes
        if nf == 0:
            return True
        sx, sy = self.node_size_x[n - nf:], self.node_size_y[n - nf:]
        return bool((sx == sx[0]).all().item() and (sy == sy[0]).all().item())

    def reorder_fillers(self, perm=None, origin_offset=(0.0, 0.0), extra=()):
        """Relabel the fillers so that those in one 64x64-bin tile of the
        density kernels are consecutive: the tiled scatter's records and the
        field gather's gradient stores then run in node order instead of
        scattering.  Fillers are interchangeable (one size, no pins), so the
        objective is unchanged and each filler's gradient moves with it.
        `perm` (filler-relative, new slot -> old slot) defaults to the tile
        order of the current positions (plus origin_offset, the density
        kernels' stretch of the fillers' origin).  Applies it to `pos` and to
        the [2N] vectors in `extra` (in the same passes), keeps the
        accumulated relabelling in `filler_perm` (slot -> generated filler)
        and returns `perm` for the caller's other per-node vectors
        (permute_fillers_)."""
        n, nf = self.num_nodes, self.num_filler_nodes
        if nf == 0:
            return None
        if not self.uniform_fillers():
            raise ValueError("reorder_fillers: fillers of different sizes are not interchangeable")
        if perm is None:
            if self.pos.is_cuda:
                keys, _ = filler_tile_keys_device(self.pos, n, nf, self.xl, self.yl,
                                                  self.bin_size_x, self.bin_size_y,
                                                  self.num_bins_x, self.num_bins_y, origin_offset,
                                                  counts=False)
                perm = torch.argsort(keys, stable=True)
            else:
                perm = filler_tile_order(self.pos, n, nf, self.xl, self.yl, self.bin_size_x,
                                         self.bin_size_y, self.num_bins_x, self.num_bins_y,
                                         origin_offset)
        else:
            perm = torch.as_tensor(perm)
            if perm.numel() != nf or not torch.equal(torch.sort(perm.long().cpu()).values,
                                                     torch.arange(nf)):
                raise ValueError("reorder_fillers: perm must be a permutation of the %d fillers" % nf)
        perm = perm.to(device=self.device, dtype=torch.int64)
        permute_fillers_many_([self.t["pos"]] + list(extra), n, nf, perm)
        fp = self.__dict__.get("filler_perm")
        self.filler_perm = perm.clone() if fp is None else fp[perm]
        return perm

    def reorder_movables(self, order):
        """Relabel the movable cells: cell i becomes the current cell
        order[i] (a permutation of [0, num_movable_nodes)).  Pins keep their
        ids and each net its pin order; each cell keeps its pins in their CSR
        order.  Every sum of the objective (per net in pin order, per node in
        CSR order, the integer density map) then keeps its terms and their
        order: the objective is the same bits and each cell's gradient moves
        with it.  For set-up, before objectives or optimizer state exist.
        The accumulated relabelling is kept in `movable_perm` (slot ->
        generated cell)."""
        m, n, dev = self.num_movable_nodes, self.num_nodes, self.device
        if m == 0:
            return  # nothing to relabel
        order = torch.as_tensor(order).to(device=dev, dtype=torch.int64)
        if order.numel() != m or not torch.equal(torch.sort(order).values,
                                                 torch.arange(m, device=dev)):
            raise ValueError("reorder_movables: order must be a permutation of the %d movable cells" % m)
        inv = torch.empty_like(order)
        inv[order] = torch.arange(m, device=dev)
        p = self.t["pos"].view(2, n)
        p[:, :m] = p[:, :m][:, order]
        for k in ("node_size_x", "node_size_y"):
            self.t[k][:m] = self.t[k][:m][order]
        if "movable_macro_mask" in self.t:
            self.t["movable_macro_mask"] = self.t["movable_macro_mask"][order].contiguous()
        remap = lambda a: torch.where(a < m, inv[a.clamp(max=m - 1)], a).to(torch.int32)
        if "sorted_node_map" in self.t:
            self.t["sorted_node_map"] = remap(self.t["sorted_node_map"].long())
        self.t["pin2node_map"] = remap(self.t["pin2node_map"].long())
        st = self.t["flat_node2pin_start_map"].long()
        nphys = st.numel() - 1
        old_of_new = torch.cat([order, torch.arange(m, nphys, device=dev)])
        lens = st[old_of_new + 1] - st[old_of_new]
        nst = torch.zeros(nphys + 1, dtype=torch.int64, device=dev)
        nst[1:] = torch.cumsum(lens, 0)
        idx = (torch.repeat_interleave(st[old_of_new] - nst[:-1], lens)
               + torch.arange(int(nst[-1].item()), device=dev))
        self.t["flat_node2pin_map"] = self.t["flat_node2pin_map"][idx].contiguous()
        self.t["flat_node2pin_start_map"] = nst.to(torch.int32)
        mp = self.__dict__.get("movable_perm")
        self.movable_perm = order.clone() if mp is None else mp[order]

    def current_order(self, v):
        """A copy of a [2N] per-node vector given in the generation order,
        with the movable cells and the fillers in the current order."""
        out = v.clone()
        mp = self.__dict__.get("movable_perm")
        if mp is not None:
            n, m = self.num_nodes, self.num_movable_nodes
            out.view(2, n)[:, :m] = v.view(2, n)[:, :m][:, mp]
        fp = self.__dict__.get("filler_perm")
        if fp is not None:
            permute_fillers_(out, self.num_nodes, self.num_filler_nodes, fp)
        return out

    def generation_order(self, v):
        """A copy of a [2N] per-node vector with the movable cells and the
        fillers back in the order the design was generated in."""
        fp = self.__dict__.get("filler_perm")
        mp = self.__dict__.get("movable_perm")
        n, nf, m = self.num_nodes, self.num_filler_nodes, self.num_movable_nodes
        out = v.clone()
        if fp is not None:
            out.view(2, n)[:, n - nf:][:, fp] = v.view(2, n)[:, n - nf:]
        if mp is not None:
            out.view(2, n)[:, :m][:, mp] = v.view(2, n)[:, :m]
        return out

    def host_design(self, like):
        """A host design dict (the layout of `like`, the dict this design was
        made from) holding this design's arrays in their current order: the
        relabelled positions, sizes and netlist maps together, each array in
        the dtype it has in `like`.  What another form of the same placement
        (another precision, a CPU run) is built from."""
        out = type(like)(like)
        for k, v in like.items():
            if isinstance(v, np.ndarray):
                out[k] = self.t[k].cpu().numpy().astype(v.dtype, copy=False)
        return out

    def __getattr__(self, k):
        t = self.__dict__.get("t", {})
        if k in t:
            return t[k]
        s = self.__dict__.get("scalars", {})
        if k in s:
            return s[k]
        raise AttributeError(k)


def filler_tile_keys(pos, num_nodes, num_fillers, xl, yl, bin_size_x, bin_size_y, num_bins_x,
                     num_bins_y, origin_offset=(0.0, 0.0), tile=64):
    """Tile of each filler's lower-left bin, tile-major as the tiled density
    kernels number tiles, for the origin pos + origin_offset (the stretched
    origin the kernels bin, in their operation order: (x + ox - xl) / bin)."""
    n, f0 = int(num_nodes), int(num_nodes) - int(num_fillers)
    x, y = pos[f0:n], pos[n + f0:2 * n]
    ox, oy = origin_offset
    bx = torch.floor((x + ox - xl) * (1.0 / bin_size_x)).clamp_(0, num_bins_x - 1).to(torch.int64)
    by = torch.floor((y + oy - yl) * (1.0 / bin_size_y)).clamp_(0, num_bins_y - 1).to(torch.int64)
    nty = (int(num_bins_y) + tile - 1) // tile
    return (bx // tile) * nty + by // tile


def filler_tile_order(pos, num_nodes, num_fillers, xl, yl, bin_size_x, bin_size_y, num_bins_x,
                      num_bins_y, origin_offset=(0.0, 0.0), tile=64):
    """Filler-relative permutation (new slot -> old slot) that sorts the
    fillers by filler_tile_keys; stable, so fillers within a tile keep their
    relative order."""
    return torch.argsort(filler_tile_keys(pos, num_nodes, num_fillers, xl, yl, bin_size_x,
                                          bin_size_y, num_bins_x, num_bins_y, origin_offset, tile),
                         stable=True)


def permute_fillers_(v, num_nodes, num_fillers, perm):
    """In place: v's filler entries (both halves of a [2N] vector) take the
    order perm (filler-relative, new slot -> old slot)."""
    permute_fillers_many_([v], num_nodes, num_fillers, perm)


def permute_fillers_many_(vectors, num_nodes, num_fillers, perm):
    """permute_fillers_ for several [2N] vectors: on the device one gather
    and one store pass per four vectors (dp_permute_fillers, bit-identical
    to the indexing below, which host tensors take)."""
    n, nf = int(num_nodes), int(num_fillers)
    vectors = [v for v in vectors if v is not None]
    if nf == 0 or not vectors:
        return
    if not vectors[0].is_cuda:
        f0 = n - nf
        for v in vectors:
            v2 = v.view(2, n)
            v2[:, f0:] = v2[:, f0:][:, perm]
        return
    perm = perm.to(device=vectors[0].device, dtype=torch.int64).contiguous()
    for k0 in range(0, len(vectors), 4):
        group = vectors[k0:k0 + 4]
        dt = group[0].dtype
        for v in group:
            if v.dtype != dt or v.numel() != 2 * n or not v.is_contiguous() or not v.is_cuda:
                raise ValueError("permute_fillers_many_: contiguous [2N] device vectors of one dtype")
        code = N.dtype_code(group[0])
        ws = torch.empty(N.query("dp_permute_fillers_workspace_bytes", code, nf, len(group)),
                         dtype=torch.uint8, device=group[0].device)
        ptrs = (N.ctypes.c_void_p * len(group))(*[v.data_ptr() for v in group])
        N.call("dp_permute_fillers", code, ptrs, len(group), n, nf, N.ptr(perm), N.ptr(ws),
               N.stream_ptr(group[0].device))


def filler_tile_keys_device(pos, num_nodes, num_fillers, xl, yl, bin_size_x, bin_size_y,
                            num_bins_x, num_bins_y, origin_offset=(0.0, 0.0), counts=True):
    """filler_tile_keys on the device in one pass (dp_filler_tile_keys): the
    same keys as int16, and with `counts` the fillers per tile (int32)."""
    n, nf = int(num_nodes), int(num_fillers)
    ntiles = ((int(num_bins_x) + 63) // 64) * ((int(num_bins_y) + 63) // 64)
    keys = torch.empty(max(nf, 1), dtype=torch.int16, device=pos.device)[:nf]
    cnt = torch.empty(ntiles, dtype=torch.int32, device=pos.device) if counts else None
    ox, oy = origin_offset
    N.call("dp_filler_tile_keys", N.dtype_code(pos), N.ptr(pos.contiguous()), n, nf, float(xl),
           float(yl), float(bin_size_x), float(bin_size_y), int(num_bins_x), int(num_bins_y),
           float(ox), float(oy), N.ptr(keys), N.ptr(cnt), N.stream_ptr(pos.device))
    return keys, cnt


def check_netlist(flat_netpin, netpin_start, pin2net, flat_node2pin, node2pin_start, num_pins,
                  num_physical_nodes):
    """Host check of the netlist maps the pin-parallel kernels index with:
    both flat maps are permutations of [0, P), the CSR starts are monotone and
    cover [0, P), and pin2net agrees with the net CSR.  Raises ValueError."""
    P = int(num_pins)
    for name, perm in (("flat_net2pin_map", flat_netpin), ("flat_node2pin_map", flat_node2pin)):
        if len(perm) != P or not np.array_equal(np.sort(perm), np.arange(P, dtype=perm.dtype)):
            raise ValueError("%s is not a permutation of [0, num_pins)" % name)
    for name, st, n in (("flat_net2pin_start_map", netpin_start, None),
                        ("flat_node2pin_start_map", node2pin_start, num_physical_nodes)):
        st = np.asarray(st, dtype=np.int64)
        if n is not None and len(st) < n + 1:
            raise ValueError("%s has fewer than num_physical_nodes+1 entries" % name)
        st = st if n is None else st[:n + 1]
        if st[0] != 0 or st[-1] != P or np.any(np.diff(st) < 0):
            raise ValueError("%s is not a CSR start array over [0, num_pins)" % name)
    deg = np.diff(np.asarray(netpin_start, dtype=np.int64))
    owner = np.repeat(np.arange(len(deg)), deg)
    if not np.array_equal(np.asarray(pin2net)[np.asarray(flat_netpin)], owner):
        raise ValueError("pin2net_map disagrees with flat_net2pin_map / flat_net2pin_start_map")




def can_track_metrics(schedule, algorithm, num_bins_x, num_bins_y, padding, uniform_fillers):
    """Whether PlacementObjective(track_metrics=True) applies: the pins
    schedule, the tiled density algorithm within its tile limit, no padding
    and fillers of one size (or none)."""
    tiles = ((int(num_bins_x) + 63) // 64) * ((int(num_bins_y) + 63) // 64)
    return (schedule == "pins" and algorithm == "tiled" and tiles <= MAX_TILES
            and int(padding) == 0 and bool(uniform_fillers))


# Pins from which the wirelength forward takes the second stream: the fork and
# join cost about 15 us of host time per evaluation.  Measured, two streams /
# one, FP32: 43 thousand pins 103 / 69 us, 1.1 million 146 / 132, 1.8 million
# 150 / 143, 3.1 million 192 / 178, 5.2 million 386 / 410, 9.6 million 433 / 467;
# FP64: 106 / 73, 604 thousand 114 / 107, 3.1 million 266 / 281, 5.2 million
# 651 / 637.  (A rule on pins and cells together, which takes two streams for 1.2
# million pins with 11 million fillers, gave 280 there for 276.)  In FP64 neither
# way is the quicker throughout from 0.6 to 5.2 million pins, by 2 to 6%.
OVERLAP_MIN_PINS = 1 << 22

# Pins from which the pins schedule permutes between node and net order in
# tiles (dp_wa_forward_tiles) instead of storing each pin's word to its place:
# below, the words of a tile are few and all of both orders stays in L2.
# Measured per evaluation, tiles / direct, FP32: 43 thousand pins 75 / 69 us,
# 433 thousand 88 / 89, 1.1 million 132 / 147, 3.1 million 178 / 229, 5.2 million
# 386 / 518, 9.6 million 433 / 700; FP64: 433 thousand 100 / 101, 1.1 million
# 179 / 197, 5.2 million 637 / 706.
TILE_MIN_PINS = 1 << 19


def net_tiles(cap, start, slices, node_dst, slot_meta):
    """The tiles and places of dp_wa_forward_tiles (see there) for tiles of at
    most `cap` cells, or None where they do not apply (exchange.node_tiles).
    start: the nodes' CSR start array; slices: of pack_slices; node_dst, slot_meta: of dp_wa_slices_prepare.  `big_shift` is a big net's
    first place - its first slot."""
    first_slot = np.concatenate([[0], 64 * np.cumsum(slices[:, 1] & 255, dtype=np.int64)])
    big0 = int(first_slot[-1])
    size = exchange.tile_size(big0, cap, 256)
    x = exchange.node_tiles(cap, start)
    if x is None or size is None:
        return None
    # tile k: the slices that begin in [k size, (k + 1) size)
    nets = np.searchsorted(first_slot, np.arange(-(-big0 // size) + 1) * size)
    nets[-1] = len(slices)
    nt = len(nets) - 1
    slots = node_dst.long()                      # node-order slot -> slot
    in_slice = slots < big0
    small = int(in_slice.sum())
    # the net tile of each pin; nets above 64 pins count as further tiles
    tile_slot = torch.from_numpy(first_slot[nets]).to(slots.device)
    t = torch.searchsorted(tile_slot, slots, right=True) - 1
    t = torch.where(in_slice, t, nt + (slots - big0) // cap)
    place = torch.empty_like(slots)
    by_net = torch.sort(t, stable=True).indices
    place[by_net] = torch.arange(len(slots), device=slots.device)
    place = torch.where(in_slice, place, small + slots - big0)
    place_of = torch.searchsorted(t[by_net].contiguous(), torch.arange(nt + 1, device=t.device))
    # a net above 64 pins has no cell; its pins follow the tiles' places
    masked = slot_meta[slots] < 0
    cell = torch.where(in_slice, slots - tile_slot[t.clamp(max=nt)], 0)
    x.update(exchange.places(x, t, place, cell, place_of[:-1] if small == len(slots)
                             else place_of, masked))
    by_place = torch.empty_like(masked)
    by_place[place] = masked
    x["big_meta"] = (x.pop("place") - (by_place.long() << 31))[small:].int()
    x.update(net_tiles=torch.stack([torch.from_numpy(nets).to(t.device), place_of],
                                   1).int().contiguous(), first_big=small, big_shift=-big0)
    return x


class PinPlan:
    """Static plan of the wirelength pass for a netlist: nets sorted by degree
    into slices of 64 (dp_wa_pack_slices), the nets above 64 pins, and the
    node-order pin offsets, destinations and slice-order metadata of
    dp_wa_slices_prepare."""

    def __init__(self, dd):
        start = dd.flat_net2pin_start_map.cpu().numpy().astype(np.int32)
        P = dd.num_pins
        check_netlist(dd.flat_net2pin_map.cpu().numpy(), start, dd.pin2net_map.cpu().numpy(),
                      dd.flat_node2pin_map.cpu().numpy(), dd.flat_node2pin_start_map.cpu().numpy(),
                      P, dd.num_physical_nodes)
        slices, lanes, big, net_slot, slots = pack_slices(start)
        self.num_slices, self.num_big, self.num_nets = len(slices), len(big), len(start) - 1
        self.num_slots = slots
        dev = dd.device
        # one copy to the device, the widest words first
        host = [big, lanes, slices, net_slot]
        parts = torch.from_numpy(np.concatenate([a.ravel() for a in host])).to(dev).split(
            [a.size for a in host])
        self.big, self.lane_nets, self.slices = [t.view(-1, k) for t, k in zip(parts, (4, 2, 2))]
        net_slot_d = parts[3]
        code = N.dtype_code(dd.pos)
        self.node_offsets = torch.empty(2 * P, dtype=dd.dtype, device=dev)
        self.node_dst = torch.empty(P, dtype=torch.int32, device=dev)
        self.slot_node = torch.empty(P, dtype=torch.int32, device=dev)
        self.slot_meta = torch.zeros(slots, dtype=torch.int32, device=dev)
        prep_ws = torch.empty(N.query("dp_wa_prepare_workspace_bytes", P), dtype=torch.uint8,
                              device=dev)
        self.tiles = None
        pin_mask = dd.pin_mask_ignore_fixed_macros
        N.call("dp_wa_slices_prepare", code, P, dd.num_physical_nodes, N.ptr(dd.pin_offset_x),
               N.ptr(dd.pin_offset_y), N.ptr(dd.flat_net2pin_map), N.ptr(dd.flat_net2pin_start_map),
               N.ptr(dd.pin2net_map), N.ptr(pin_mask), N.ptr(dd.flat_node2pin_map),
               N.ptr(dd.flat_node2pin_start_map), N.ptr(net_slot_d), N.ptr(prep_ws),
               N.ptr(self.node_offsets), N.ptr(self.node_dst), N.ptr(self.slot_node),
               N.ptr(self.slot_meta), N.stream_ptr(dev))
        del net_slot_d
        del prep_ws  # stream-ordered: the caching allocator reuses it only after the kernels
        if P >= TILE_MIN_PINS:
            self.tiles = net_tiles(
                N.query("dp_wa_tile_pins", code),
                dd.flat_node2pin_start_map[:dd.num_physical_nodes + 1], slices, self.node_dst,
                self.slot_meta)
        if self.tiles is not None:
            self.big[:, 1] += self.tiles["big_shift"]
            self.node_offsets = self.node_offsets.view(P, 2)[self.tiles.pop("slot_of")].view(-1)
            del self.node_dst, self.slot_node, self.slot_meta
        self.ws = torch.empty(N.query("dp_wa_pins_workspace_bytes",
                                      slots if self.tiles is None else P, code),
                              dtype=torch.uint8, device=dev)
        self.num_partials = N.query("dp_wa_num_partials", self.num_slices, 0 if self.tiles is None
                                    else len(self.tiles["net_tiles"]) - 1, self.num_big)
        # each pin's derivative, in node order or in the exchange's
        self.pin_grad = torch.empty(2 * P, dtype=dd.dtype, device=dev)


class PlacementObjective:
    def __init__(self, dd, gamma, density_weight=1.0, precision=None, fused=True,
                 energy_mode="potential", convention="cpu", algorithm="global", schedule=None,
                 keep_partial_wl=False, wirelength="weighted_average", overlap=True,
                 track_metrics=False, density_backward="force", wa_arith="reference",
                 density_arith="reference"):
        """keep_partial_wl: also store the per-net (pre-weight) wirelength in
        `partial_wl` (what the net-weight adjoint needs); the pins schedule
        skips that store otherwise.  wirelength: "weighted_average" or
        "logsumexp" (PlaceObj.py:467-503); the log-sum-exp model runs on the
        "pins" and "unfused" schedules.  overlap (pins schedule): run the
        wirelength forward of a netlist of OVERLAP_MIN_PINS pins or more on a
        second stream, concurrently with the density chain it does not depend
        on; the node-gradient pass joins them.
        track_metrics (pins schedule, tiled density, fillers of one size, no
        padding): every evaluation also leaves the placer's metrics at its
        positions in `metric_out` (FP64 {HPWL, overflow cost, max bin
        density}): the HPWL from the wirelength pass's per-net extremes, the
        overflow from the same scatter's fixed + movable map.  Both are
        bit-identical to dp_hpwl and to ElectricOverflow's own scatter.
        `metric_ptr` is the address of those positions; a caller that changes
        them in place clears it.  density_backward: "force" (the reference's
        field gather) or "adjoint" (the exact derivative of the energy,
        dp_energy_gradient, from the potential map the solve then writes).
        wa_arith (pins schedule, weighted average): "reference" evaluates the
        reference's merged (a + b x) e derivative; "centred" the same model
        relative to each net's extremes (DP_WL_WEIGHTED_AVERAGE_CENTRED), which
        keeps FP32 near its rounding level instead of ~2e-5.  density_arith:
        "reference" or "bin_relative" overlaps in the density scatter, the
        fixed map and the field gather (ElectricPotential's `arithmetic`)."""
        if wa_arith not in ("reference", "centred"):
            raise ValueError("wa_arith must be 'reference' or 'centred', got %r" % (wa_arith,))
        self.wa_arith = wa_arith
        if density_backward not in ("force", "adjoint"):
            raise ValueError("density_backward must be 'force' or 'adjoint', got %r"
                             % (density_backward,))
        self.density_backward = density_backward
        if wirelength not in ("weighted_average", "logsumexp"):
            raise ValueError("wirelength must be weighted_average or logsumexp, got %r" % (wirelength,))
        self.lse = wirelength == "logsumexp"
        if self.lse and (schedule or ("fused" if fused else "unfused")) == "fused":
            raise NotImplementedError("the log-sum-exp wirelength runs on the pins or unfused schedule")
        self.dd = dd
        self.keep_partial_wl = keep_partial_wl
        dt = dd.dtype
        dev = dd.device
        self.fused = fused
        # schedule: "pins" (pin-parallel WA + contiguous node backward),
        # "fused" (net-parallel fused kernels) or "unfused" (reference op order)
        self.schedule = schedule or ("fused" if fused else "unfused")
        self.pin_plan = PinPlan(dd) if self.schedule == "pins" else None
        if wa_arith == "centred" and (self.lse or self.schedule != "pins"):
            raise NotImplementedError("the centred WA arithmetic runs on the pins schedule "
                                      "with the weighted-average model")
        self._wa_model = (N.DP_WL_LOGSUMEXP if self.lse else
                          N.DP_WL_WEIGHTED_AVERAGE_CENTRED if wa_arith == "centred" else
                          N.DP_WL_WEIGHTED_AVERAGE)
        self.density = ElectricPotential(
            dd.node_size_x, dd.node_size_y, dd.bin_center_x, dd.bin_center_y, dd.target_density,
            dd.xl, dd.yl, dd.xh, dd.yh, dd.bin_size_x, dd.bin_size_y, dd.num_movable_nodes,
            dd.num_terminals, dd.num_filler_nodes, 0, True, dd.sorted_node_map,
            movable_macro_mask=dd.movable_macro_mask, precision=precision,
            energy_mode=energy_mode, convention=convention, algorithm=algorithm,
            arithmetic=density_arith)
        self.density.compute_initial_density_map(dd.pos)
        self.plan = self.density.plan(dt, dev)
        self.solve_ws = self.plan.scratch()
        n, P, E = dd.num_nodes, dd.num_pins, dd.num_nets
        M, Nb = self.density.num_bins_x, self.density.num_bins_y
        z = lambda *s, dtype=dt: torch.empty(*s, dtype=dtype, device=dev)
        self.inv_gamma = torch.tensor(1.0 / gamma, dtype=dt, device=dev)
        self.gamma_t = torch.tensor(float(gamma), dtype=dt, device=dev)
        self.lam = torch.tensor(float(density_weight), dtype=dt, device=dev)
        self.lam_host = float(density_weight)
        self.density_factor = 1.0
        self.quad_coeff = None
        self.lam_eff = torch.empty((), dtype=dt, device=dev)
        self.one = torch.ones((), dtype=dt, device=dev)
        self.wl = z(())
        self.partial_wl = z(E)
        self.grad_intermediate = torch.zeros(2 * P, dtype=dt, device=dev)
        self.pin_pos = z(2 * P)
        self.density_map = z(M, Nb)
        pdt = self.plan.dtype
        self.field_x = torch.empty(M, Nb, dtype=pdt, device=dev)
        self.field_y = torch.empty_like(self.field_x)
        self.potential = (torch.empty_like(self.field_x)
                          if energy_mode == "potential" or density_backward == "adjoint" else None)
        self.energy = torch.empty((), dtype=pdt, device=dev)
        # the pins schedule keeps the density gradient interleaved ((x, y) per
        # node: one scattered word per cell in the gather); others keep [2N]
        self.grad_layout = N.DP_LAYOUT_INTERLEAVED if self.schedule == "pins" else N.DP_LAYOUT_SPLIT
        self._density_grad = z(2 * n)
        self.wl_grad = z(2 * n)
        self.grad = z(2 * n)
        self.obj = z(())
        self.wa_ws = torch.empty(N.query("dp_wa_workspace_bytes", E), dtype=torch.uint8, device=dev)
        self.w = dd.net_weights.contiguous()
        self.net_mask = dd.net_mask_ignore_large_degrees
        self.pin_mask = dd.pin_mask_ignore_fixed_macros
        # a second stream (default priority) for the wirelength forward
        self.side = None
        self._side_stream = None
        # where the wirelength pass forks off: before the scatter ("scatter"),
        # "solve" or "gather".  With the kernels of then, 9.6 million pins and 13
        # million cells: 0.729 ms, 0.750 before the solve, 0.736 before the
        # gather, 0.766-0.770 on one stream; 53 million cells: 1.494, 1.524,
        # 1.547, 1.498-1.507
        self.fork_at = "scatter"
        self.set_overlap(overlap)
        self.filler_ranges = None
        self._dg2 = None
        self._norm_ws = None
        self.last_dg2 = None
        self.track_metrics = False
        self.metric_ptr = None
        if track_metrics:
            ep = self.density
            if not can_track_metrics(self.schedule, ep.algorithm, M, Nb, ep.padding,
                                     dd.num_filler_nodes == 0 or ep.use_uniform_filler):
                raise ValueError("track_metrics needs the pins schedule, the tiled density "
                                 "algorithm (at most %d tiles), no padding and fillers of one size"
                                 % MAX_TILES)
            self.track_metrics = True
            self.net_hpwl = z(E)
            self.movable_map = z(M, Nb)
            self.metric_out = torch.empty(3, dtype=torch.float64, device=dev)
            self.metric_ws = torch.empty(N.query("dp_step_metrics_workspace_bytes"),
                                         dtype=torch.uint8, device=dev)
        # the fillers' gradient combine (and preconditioner) done by the field
        # gather itself (dp_electric_force_fillers_final): the same bits, one
        # pass over the fillers fewer; where it applies (pins schedule, tiled
        # gather, fillers of one size, the reference's force backward)
        ep = self.density
        self.fillers_final = (dd.num_filler_nodes > 0 and density_backward != "adjoint"
                              and can_track_metrics(self.schedule, ep.algorithm, M, Nb,
                                                    ep.padding, ep.use_uniform_filler))
        self._ff_last = None  # (gradient buffer, preconditioned) of the last evaluation

    def filler_origin_offset(self):
        """The stretch offset of the fillers' origin in the density kernels
        (one value for fillers of one size), for sorting them by tile."""
        ep = self.density
        uf = ep.uniform_filler if ep.use_uniform_filler else None
        return (uf[2], uf[3]) if uf else (0.0, 0.0)

    def update_filler_ranges(self, pos):
        """After the caller has put the fillers in tile order
        (DeviceDesign.reorder_fillers with filler_origin_offset()): the
        per-tile filler ranges the tiled scatter and gather then take instead
        of binning the fillers (dp_density_map_ex).  Positions may move
        afterwards; results stay exact, speed falls as fillers leave their
        tiles.  Returns False, using none, where they do not apply (not the
        tiled algorithm, fillers of several sizes or stretched past 2 bins)."""
        ep, dd = self.density, self.dd
        uf = ep.uniform_filler if ep.use_uniform_filler else None
        nf = dd.num_filler_nodes
        self.filler_ranges = None
        if (ep.algorithm != "tiled" or nf == 0 or uf is None or uf[0] > 1.99 * ep.bin_size_x
                or uf[1] > 1.99 * ep.bin_size_y):
            return False
        M, Nb = ep.num_bins_x, ep.num_bins_y
        ntiles = ((M + 63) // 64) * ((Nb + 63) // 64)
        _, counts = filler_tile_keys_device(pos, dd.num_nodes, nf, float(ep.xl), float(ep.yl),
                                            float(ep.bin_size_x), float(ep.bin_size_y), M, Nb,
                                            (uf[2], uf[3]))
        fr = torch.zeros(ntiles + 1, dtype=torch.int32, device=pos.device)
        fr[1:] = torch.cumsum(counts, 0)
        self.filler_ranges = fr
        return True

    def set_overlap(self, on):
        """Run the pins schedule's wirelength forward on a second stream
        (on=True; from OVERLAP_MIN_PINS pins on, below which that is slower and
        it keeps to the caller's) or on the caller's stream.  Either gives the
        same bits."""
        if on and self.schedule == "pins":
            if self._side_stream is None:
                self._side_stream = torch.cuda.Stream(device=self.dd.device)
                self._side_handle = self._side_stream.cuda_stream
                self._ev_fork = torch.cuda.Event()
                self._ev_join = torch.cuda.Event()
            self.side = self._side_stream
        else:
            self.side = None

    @property
    def overlap(self):
        """Whether the second stream is switched on (set_overlap)."""
        return self.side is not None

    def set_net_weights(self, w):
        """New per-net weights (e.g. from timing-driven net weighting)."""
        self.w = w.to(self.dd.dtype).contiguous()

    @property
    def density_grad(self):
        """Density gradient of the last evaluation in the reference [2N] layout.
        Where the field gather finished the fillers' gradients itself, theirs
        are read back from that evaluation's gradient buffer (0 + g: the same
        values, a negative zero read as zero), which must not have been
        written since; not available after a preconditioned evaluation, whose
        filler gradients are divided (set `fillers_final = False` before an
        evaluation whose density gradient is wanted in full)."""
        if self.grad_layout == N.DP_LAYOUT_INTERLEAVED:
            g = self._density_grad.view(-1, 2).t().reshape(-1)
        else:
            g = self._density_grad
        if self._ff_last is not None:
            buf, pre = self._ff_last
            if pre:
                raise RuntimeError("density_grad: the last evaluation was preconditioned and "
                                   "kept only the fillers' finished gradients")
            n = self.dd.num_nodes
            f0 = n - self.dd.num_filler_nodes
            if g.data_ptr() == self._density_grad.data_ptr():
                g = g.clone()
            g[f0:n] = buf[f0:n]
            g[n + f0:] = buf[n + f0:]
        return g

    def set_gamma(self, gamma):
        self.inv_gamma.fill_(1.0 / gamma)
        self.gamma_t.fill_(float(gamma))

    def set_density_weight(self, w):
        self.lam_host = float(w)
        self.lam.fill_(float(w))

    def set_density_penalty(self, factor=1.0, quad_coeff=None):
        """PlaceObj.obj_fn's penalty forms (dreamplace/PlaceObj.py:293-320):
        obj = WL + (factor * lambda) * D, or with the quadratic penalty
        obj = WL + (factor * lambda) * D * (1 + c * D), c = quad_coeff."""
        self.density_factor = float(factor)
        self.quad_coeff = None if quad_coeff is None else float(quad_coeff)

    # -- stages ---------------------------------------------------------------
    def _density_forward(self, pos):
        self._density_scatter(pos)
        self._density_solve()

    def _density_scatter(self, pos):
        ep = self.density
        N.call("dp_density_map_ex", N.dtype_code(pos), N.ptr(pos), pos.numel() // 2,
               N.ptr(ep.node_size_x_clamped), N.ptr(ep.node_size_y_clamped), N.ptr(ep.offset_x),
               N.ptr(ep.offset_y), N.ptr(ep.ratio), N.ptr(ep.initial_density_map), float(ep.xl),
               float(ep.yl), float(ep.xh), float(ep.yh), float(ep.bin_size_x),
               float(ep.bin_size_y), int(ep.num_movable_nodes), int(ep.num_filler_nodes),
               ep.num_bins_x, ep.num_bins_y,
               N.DP_CONVERT_CPU if ep.convention == "cpu" else N.DP_CONVERT_GPU,
               ep.run_code(), ep.large_capacity, ep.uniform_filler_arg(),
               N.ptr(self.filler_ranges), N.ptr(ep.workspace(pos.device)),
               N.ptr(self.density_map), N.ptr(self.movable_map) if self.track_metrics else None,
               N.stream_ptr(pos.device))

    def _density_solve(self):
        ep = self.density
        dmap = self.density_map
        if dmap.dtype != self.plan.dtype:
            dmap = dmap.to(self.plan.dtype)
        want_energy = not ep.fast_mode
        self.plan.poisson(dmap, ep.bin_size_x, ep.bin_size_y,
                          compute_potential=self.potential is not None
                          and (want_energy or self.density_backward == "adjoint"),
                          compute_energy=want_energy,
                          out=(self.field_x, self.field_y, self.potential, self.energy),
                          ws=self.solve_ws)

    def _reduce_metrics(self, pos, s):
        """metric_out = {HPWL (design net weights, all nets of two or more
        pins), overflow cost, max bin density} at `pos`, from this
        evaluation's per-net extremes and fixed + movable map."""
        dd, ep = self.dd, self.density
        bin_area = float(ep.bin_size_x) * float(ep.bin_size_y)
        N.call("dp_step_metrics", N.dtype_code(self.net_hpwl), N.ptr(self.net_hpwl),
               N.ptr(dd.flat_net2pin_start_map), dd.num_nets, N.ptr(dd.net_weights),
               N.ptr(dd.net_mask_all), N.ptr(self.movable_map), self.movable_map.numel(),
               float(ep.target_density) * bin_area, N.ptr(self.metric_ws), N.ptr(self.metric_out),
               s)
        self.metric_ptr = pos.data_ptr()

    def _energy(self, pos):
        e = self.energy
        return e if e.dtype == pos.dtype else e.to(pos.dtype)

    def _density_grad_weight(self, pos):
        """d obj / d D on the device: factor * lambda, times (1 + c D) +
        D c under the quadratic penalty (the product rule's two terms, in
        autograd's order)."""
        if self.quad_coeff is None and self.density_factor == 1.0:
            return self.lam
        g = torch.mul(self.lam, self.density_factor, out=self.lam_eff)
        if self.quad_coeff is not None:
            e = self._energy(pos)
            c = self.quad_coeff
            self.lam_eff.copy_(g * (1 + c * e) + (g * e) * c)
        return self.lam_eff

    def _density_backward(self, pos, ff=None):
        """ff: (gradient buffer, density weight or None, alpha, filler area)
        for dp_electric_force_fillers_final, else None."""
        ep = self.density
        w = self._density_grad_weight(pos)
        if self.density_backward == "adjoint":
            phi = self.potential if self.potential.dtype == pos.dtype else self.potential.to(pos.dtype)
            N.call("dp_energy_gradient", N.dtype_code(pos), N.ptr(w), N.ptr(phi), N.ptr(pos),
                   pos.numel() // 2, N.ptr(ep.node_size_x_clamped), N.ptr(ep.node_size_y_clamped),
                   N.ptr(ep.offset_x), N.ptr(ep.offset_y), N.ptr(ep.ratio), float(ep.xl),
                   float(ep.yl), float(ep.bin_size_x), float(ep.bin_size_y),
                   int(ep.num_movable_nodes), int(ep.num_filler_nodes), ep.num_bins_x,
                   ep.num_bins_y, self.grad_layout, ep.uniform_filler_arg(),
                   N.ptr(self._density_grad), N.stream_ptr(pos.device))
            return
        fx, fy = self.field_x, self.field_y
        if fx.dtype != pos.dtype:
            fx, fy = fx.to(pos.dtype), fy.to(pos.dtype)
        args = (N.dtype_code(pos), N.ptr(w), N.ptr(fx), N.ptr(fy),
                N.ptr(pos), pos.numel() // 2, N.ptr(ep.node_size_x_clamped),
                N.ptr(ep.node_size_y_clamped), N.ptr(ep.offset_x), N.ptr(ep.offset_y),
                N.ptr(ep.ratio), float(ep.xl), float(ep.yl), float(ep.bin_size_x),
                float(ep.bin_size_y), int(ep.num_movable_nodes), int(ep.num_filler_nodes),
                ep.num_bins_x, ep.num_bins_y, ep.run_code(), ep.large_capacity,
                self.grad_layout, ep.uniform_filler_arg(), N.ptr(ep.workspace(pos.device)),
                N.ptr(self._density_grad))
        if ff is None:
            N.call("dp_electric_force", *args, N.stream_ptr(pos.device))
        else:
            buf, dw, alpha, farea = ff
            N.call("dp_electric_force_fillers_final", *args, N.ptr(buf), N.ptr(dw), float(alpha),
                   float(farea), N.stream_ptr(pos.device))

    def _node_grad(self, code, layout, grad, pre, norm, s):
        """The nodes' sums of their pins' derivatives, plus the density
        gradient, preconditioned with `pre` unless that is None; the
        wirelength's total; and the objective, where it is the wirelength plus
        a weight times the solve's energy (then True)."""
        dd, pp = self.dd, self.pin_plan
        x = pp.tiles
        tiles = ((N.ptr(x["node_tiles"]), len(x["node_tiles"]) - 1, N.ptr(x["node_cell"]))
                 if x is not None else (None, 0, None))
        whole = self.quad_coeff is None and self.energy.dtype == self.obj.dtype
        N.call("dp_node_grad_objective", code, N.ptr(self.one), N.ptr(pp.pin_grad), *tiles,
               N.ptr(dd.flat_node2pin_start_map), N.ptr(self._density_grad), layout,
               dd.num_physical_nodes, dd.num_nodes, *(pre or (None, None, None, 0.0, -1.0)),
               N.ptr(grad), *norm, N.ptr(pp.ws), pp.num_partials, N.ptr(self.wl),
               N.ptr(self.energy) if whole else None, self.density_factor * self.lam_host,
               N.ptr(self.obj) if whole else None, s)
        return whole

    def evaluate(self, pos, precondition=None, grad_out=None, grad_ref=None):
        """(obj 0-dim tensor, grad [2N] tensor); both are reused buffers.
        precondition = (pin_weight_sum, node_areas, alpha[, filler_area])
        also applies PlaceObj's preconditioner to the gradient (with the
        current density weight), fused into the node-gradient pass on the pins
        schedule; filler_area >= 0 states that every filler has that area
        (and, having no pins, a zero pin-weight sum), so that pass reads
        neither array for them.
        grad_out: a contiguous [2N] tensor of the positions' type and device
        that receives the gradient (and is returned) instead of the
        objective's own buffer, so a caller that keeps gradients from step to
        step needs no copy.
        grad_ref: a [2N] gradient (not the output buffer); where the
        preconditioned node-gradient pass runs (the pins schedule) it also
        forms sum((grad - grad_ref)^2) in FP64 and leaves it in `last_dg2`
        (a device double[1]), else `last_dg2` is None."""
        grad = self.grad
        self.last_dg2 = None
        if grad_out is not None:
            if (grad_out.dtype != self.grad.dtype or grad_out.device != self.grad.device
                    or grad_out.numel() != self.grad.numel() or not grad_out.is_contiguous()):
                raise ValueError("evaluate: grad_out must be a contiguous %s tensor of %d elements on %s"
                                 % (self.grad.dtype, self.grad.numel(), self.grad.device))
            grad = grad_out
        dd = self.dd
        code = N.dtype_code(pos)
        s = N.stream_ptr(pos.device)
        n, P, E = dd.num_nodes, dd.num_pins, dd.num_nets
        self._ff_last = None
        if self.schedule == "pins":
            pp = self.pin_plan
            # the fillers' gradients finished by the field gather, where that
            # applies: unpreconditioned, or preconditioned with the fillers' area
            ff = None
            if self.fillers_final:
                if precondition is None:
                    ff = (grad, None, 0.0, -1.0)
                elif len(precondition) > 3 and precondition[3] >= 0:
                    ff = (grad, self.lam, float(precondition[2]), float(precondition[3]))
            layout = self.grad_layout | (N.DP_LAYOUT_FILLERS_FINAL if ff is not None else 0)
            # the second stream, where the netlist is large enough for it
            side = self.side if P >= OVERLAP_MIN_PINS else None

            def wirelength_forward():
                s_wl = s
                if side is not None:
                    # fork: the side stream starts after everything queued so far
                    main = torch.cuda.current_stream(pos.device)
                    self._ev_fork.record(main)
                    side.wait_event(self._ev_fork)
                    s_wl = self._side_handle
                pins = (code, self._wa_model, N.ptr(pos), n, P)
                rest = (E, N.ptr(self.w), N.ptr(self.net_mask),
                        N.ptr(self.gamma_t if self.lse else self.inv_gamma),
                        N.ptr(self.partial_wl) if self.keep_partial_wl else None,
                        N.ptr(self.net_hpwl) if self.track_metrics else None,
                        N.ptr(pp.pin_grad), None, N.ptr(pp.ws), s_wl)
                x = pp.tiles
                if x is not None:
                    N.call("dp_wa_forward_tiles", *pins, N.ptr(x["place_node"]),
                           N.ptr(pp.node_offsets), N.ptr(x["node_tiles"]),
                           len(x["node_tiles"]) - 1, N.ptr(x["node_chunk"]),
                           N.ptr(x["node_delta"]), N.ptr(x["net_tiles"]),
                           len(x["net_tiles"]) - 1, N.ptr(x["cell"]), N.ptr(x["chunk"]),
                           N.ptr(x["delta"]), N.ptr(pp.slices), N.ptr(pp.lane_nets),
                           N.ptr(pp.big), pp.num_big, N.ptr(x["big_meta"]), x["first_big"],
                           *rest)
                else:
                    N.call("dp_wa_forward_slices", *pins, N.ptr(pp.slot_node),
                           N.ptr(pp.node_offsets), N.ptr(pp.node_dst), N.ptr(pp.slot_meta),
                           N.ptr(pp.slices), N.ptr(pp.lane_nets), pp.num_slices, N.ptr(pp.big),
                           pp.num_big, *rest)
                if side is not None:
                    self._ev_join.record(side)

            # on one stream the wirelength pass goes first; with two, it forks
            # where fork_at says (the chain it overlaps is the rest)
            fork_at = self.fork_at if side is not None else "scatter"
            if fork_at == "scatter":
                wirelength_forward()
            self._density_scatter(pos)
            if fork_at == "solve":
                wirelength_forward()
            self._density_solve()
            if fork_at == "gather":
                wirelength_forward()
            self._density_backward(pos, ff)
            if ff is not None:
                self._ff_last = (grad, ff[1] is not None)
            if side is not None:
                # join: the node gradient and the objective read the wirelength outputs
                torch.cuda.current_stream(pos.device).wait_event(self._ev_join)
            if self.track_metrics:
                self._reduce_metrics(pos, s)
            if precondition is not None:
                pws, areas, alpha = precondition[:3]
                # the fillers' one area, when the caller knows it (else -1)
                farea = precondition[3] if len(precondition) > 3 else -1.0
                fuse = grad_ref is not None and grad_ref.data_ptr() != grad.data_ptr()
                if fuse and self._dg2 is None:
                    self._dg2 = torch.empty(1, dtype=torch.float64, device=pos.device)
                    self._norm_ws = torch.empty(N.query("dp_optimizer_workspace_bytes"),
                                                dtype=torch.uint8, device=pos.device)
                norm = ((N.ptr(grad_ref), N.ptr(self._norm_ws), N.ptr(self._dg2)) if fuse
                        else (None, None, None))
                pre = (N.ptr(pws), N.ptr(areas), N.ptr(self.lam), float(alpha), float(farea))
                whole = self._node_grad(code, layout, grad, pre, norm, s)
                if fuse:
                    self.last_dg2 = self._dg2
                precondition = None  # done
            else:
                whole = self._node_grad(code, layout, grad, None, (None, None, None), s)
            if whole:
                return self.obj, grad
        elif self.schedule == "fused":
            N.call("dp_wa_forward_from_nodes", code, N.ptr(pos), n, N.ptr(dd.pin_offset_x),
                   N.ptr(dd.pin_offset_y), N.ptr(dd.pin2node_map), P, N.ptr(dd.flat_net2pin_map),
                   N.ptr(dd.flat_net2pin_start_map), E, N.ptr(self.w), N.ptr(self.net_mask),
                   N.ptr(self.inv_gamma), N.ptr(self.partial_wl), N.ptr(self.grad_intermediate),
                   N.ptr(self.wl), N.ptr(self.wa_ws), s)
            self._density_forward(pos)
            self._density_backward(pos)
            N.call("dp_wa_backward_to_nodes", code, N.ptr(self.one), N.ptr(self.grad_intermediate),
                   P, N.ptr(dd.flat_node2pin_map), N.ptr(dd.flat_node2pin_start_map),
                   N.ptr(dd.pin2net_map), N.ptr(self.w), N.ptr(self.net_mask), N.ptr(self.pin_mask),
                   N.ptr(self._density_grad), dd.num_physical_nodes, n, N.ptr(grad), s)
        else:
            N.call("dp_pin_pos_forward", code, N.ptr(pos), n, N.ptr(dd.pin_offset_x),
                   N.ptr(dd.pin_offset_y), N.ptr(dd.pin2node_map), N.DP_INDEX_INT32, P,
                   N.ptr(self.pin_pos), s)
            N.call("dp_lse_merged_forward" if self.lse else "dp_wa_merged_forward", code,
                   N.ptr(self.pin_pos), P, N.ptr(dd.flat_net2pin_map),
                   N.ptr(dd.flat_net2pin_start_map), E, N.ptr(self.w), N.ptr(self.net_mask),
                   N.ptr(self.gamma_t if self.lse else self.inv_gamma), N.ptr(self.partial_wl),
                   N.ptr(self.grad_intermediate), N.ptr(self.wl), N.ptr(self.wa_ws), s)
            self._density_forward(pos)
            self._density_backward(pos)
            N.call("dp_wa_merged_backward", code, N.ptr(self.one), N.ptr(self.grad_intermediate), P,
                   N.ptr(dd.pin2net_map), N.ptr(self.w), N.ptr(self.net_mask), N.ptr(self.pin_mask),
                   s)
            N.call("dp_pin_pos_backward", code, N.ptr(self.grad_intermediate), P,
                   N.ptr(dd.flat_node2pin_map), N.ptr(dd.flat_node2pin_start_map),
                   dd.num_physical_nodes, n, N.ptr(self.wl_grad), s)
            torch.add(self.wl_grad, self._density_grad, out=grad)
        if precondition is not None:
            pws, areas, alpha = precondition[:3]
            N.call("dp_precondition", code, N.ptr(grad), n, N.ptr(pws), N.ptr(areas),
                   N.ptr(self.lam), float(alpha), s)
        energy = self._energy(pos)
        if self.quad_coeff is not None:
            energy = energy * (1 + self.quad_coeff * energy)
        torch.add(self.wl, energy, alpha=self.density_factor * self.lam_host, out=self.obj)
        return self.obj, grad
