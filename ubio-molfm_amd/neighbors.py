"""Periodic radius graph on the GPU -> query CSR + key CSR.

Semantics follow the reference's CellExpander + construct_radius_neighbor
(src/molfm/models/e2former/module_utils.py:953-988,1065-1274,3119-3242):

* shifts s with |s_d| <= min(cells_per_direction, ceil(rc / h_d)) on periodic
  dimensions (h_d = lattice height), 0 elsewhere; [0,0,0] first;
* an image (j, s) exists iff some atom of the graph is strictly within rc of it;
* edge i <- (j, s) iff rmin <= d <= rc (both inclusive);
* rows sorted by ascending distance (ties by (j, s)); ``max_neighbors`` keeps
  the nearest k of each row.

fp32 expression (identical in the kernel): off = ((s0*a) + s1*b) + s2*c per
component, img = pos_j + off, dvec = pos_i - img, d = sqrt((dx*dx + dy*dy) + dz*dz).
"""
from __future__ import annotations

import math
from collections import OrderedDict
from dataclasses import dataclass
from typing import Optional

import numpy as np
import torch

from . import _lib

F32 = np.float32
BIN_MARGIN = 1e-2


def _max_offsets(cell: np.ndarray, rc: float, cap: int):
    c = torch.as_tensor(np.asarray(cell, F32)).reshape(1, 3, 3)
    out = []
    for dim in range(3):
        lat = c[:, dim, :]
        rest = c[:, [k for k in range(3) if k != dim], :]
        nv = torch.cross(rest[:, 0, :], rest[:, 1, :], dim=-1)
        nv = nv / nv.norm(dim=-1, keepdim=True)
        try:
            out.append(int(torch.max(torch.ceil(rc / torch.abs(torch.sum(nv * lat, dim=-1))))))
        except (ValueError, RuntimeError, OverflowError):
            out.append(cap)
    return out


def shift_table(cell: np.ndarray, pbc, rc: float, cap: int = 4) -> np.ndarray:
    """Integer shifts of one graph, [0,0,0] first, then lexicographic."""
    pbc = [bool(x) for x in np.asarray(pbc).reshape(3)]
    if not any(pbc):
        return np.zeros((1, 3), np.int32)
    mo = _max_offsets(cell, rc, cap)
    rows = [(0, 0, 0)]
    for a in range(-cap, cap + 1):
        for b in range(-cap, cap + 1):
            for c in range(-cap, cap + 1):
                s = (a, b, c)
                if s == (0, 0, 0):
                    continue
                if any(abs(s[d]) > mo[d] or (s[d] != 0 and not pbc[d]) for d in range(3)):
                    continue
                rows.append(s)
    return np.asarray(rows, np.int32)


def shift_offsets(shifts: np.ndarray, cell: np.ndarray) -> np.ndarray:
    A = np.asarray(cell, F32).reshape(3, 3)
    s = shifts.astype(F32)
    return ((s[:, 0:1] * A[0] + s[:, 1:2] * A[1]) + s[:, 2:3] * A[2]).astype(F32)


@dataclass
class NeighborList:
    n_atoms: int
    n_edges: int
    row_ptr: torch.Tensor     # [N+1] int32
    col: torch.Tensor         # [E] int32 source atom
    shift_idx: torch.Tensor   # [E] int32 row of ``shifts``
    shifts: torch.Tensor      # [S,3] int32 (host)
    dvec: torch.Tensor        # [E,3] fp32
    dist: torch.Tensor        # [E] fp32
    edge_row: torch.Tensor    # [E] int32
    key_ptr: torch.Tensor     # [N+1] int32
    key_eid: torch.Tensor     # [E] int32
    max_row: int = 0
    # clusters of consecutive key-CSR columns for the attention column pass
    col_span: int = 0
    col_slot_member: Optional[torch.Tensor] = None   # [E] int32
    col_slot_edge: Optional[torch.Tensor] = None     # [E, col_span] int32
    col_n_slots: Optional[torch.Tensor] = None       # [ceil(N / col_span)] int32
    shift_ptr: Optional[np.ndarray] = None           # [B+1] rows of ``shifts`` per graph (host)
    # capacity build (build_neighbors(capacity=...)): the edge arrays hold n_edges slots of which
    # the first stats[0] are edges; stats [4] int32 on the device = {E, longest row, an atom outside
    # the grid box, overflow}; the list is valid only when stats[2] == stats[3] == 0
    stats: Optional[torch.Tensor] = None
    # ... copied without waiting to pinned host memory (stats_host), complete once stats_event has
    stats_host: Optional[torch.Tensor] = None
    stats_event: Optional[object] = None

    def canonical(self):
        """(i, j, s) sorted lexicographically, plus dvec/dist in that order (numpy)."""
        i = self.edge_row.cpu().numpy().astype(np.int64)
        j = self.col.cpu().numpy().astype(np.int64)
        s = self.shifts.numpy()[self.shift_idx.cpu().numpy()]
        dv = self.dvec.cpu().numpy()
        d = self.dist.cpu().numpy()
        o = np.lexsort((s[:, 2], s[:, 1], s[:, 0], j, i))
        return dict(i=i[o], j=j[o], s=s[o], dv=dv[o], d=d[o])


def _ptr(t: Optional[torch.Tensor]):
    return None if t is None else t.data_ptr()


def _vp(t: Optional[torch.Tensor]):
    return None if t is None or t.numel() == 0 else _lib.vp(t.data_ptr())


_PLAN_TABLES: "OrderedDict" = OrderedDict()


def _plan_tables(dev, graph_ptr, cells, pbcs, rc, cells_per_direction, bb):
    """The plan's device tables (graph pointers, shift tables and offsets, bin
    grids) and host sizes, built once per distinct input: an MD loop with a fixed
    grid box reuses them (no host-to-device copy, hence no host sync, per build)."""
    key = (str(dev), graph_ptr.tobytes(), cells.tobytes(), pbcs.tobytes(), float(rc), int(cells_per_direction),
           np.asarray(bb, F32).tobytes())
    hit = _PLAN_TABLES.get(key)
    if hit is not None:
        _PLAN_TABLES.move_to_end(key)
        return hit
    B = len(graph_ptr) - 1
    shifts, sptr, periodic = [], [0], []
    glo = np.zeros((B, 3), F32); gh = np.zeros((B, 3), F32); gdim = np.zeros((B, 3), np.int32)
    base = np.zeros(B, np.int32)
    nb = 0
    h_min = F32(rc + BIN_MARGIN)
    for g in range(B):
        sh = shift_table(cells[g], pbcs[g], rc, cells_per_direction)
        shifts.append(sh)
        sptr.append(sptr[-1] + len(sh))
        periodic.append(1 if pbcs[g].any() else 0)
        if graph_ptr[g + 1] > graph_ptr[g]:
            l, h = bb[0, g], bb[1, g]
        else:
            l, h = np.zeros(3, F32), np.zeros(3, F32)
        ext = np.maximum(h - l, 0.0)
        dims = np.maximum(1, np.floor(ext / h_min)).astype(np.int64)
        while np.prod(dims) > (1 << 22):
            dims = np.maximum(1, dims // 2)
        glo[g] = l
        gh[g] = np.maximum(ext / dims, h_min)
        gdim[g] = dims
        base[g] = nb
        nb += int(np.prod(dims))
    shifts_np = np.concatenate(shifts).astype(np.int32)
    offs = np.concatenate([shift_offsets(s, cells[g]) for g, s in enumerate(shifts)]).astype(F32)
    # the small tables in one host-to-device copy per type
    ints = [graph_ptr.astype(np.int32), np.asarray(sptr, np.int32), np.asarray(periodic, np.int32),
            gdim.reshape(-1), base, np.repeat(np.arange(B, dtype=np.int32), np.diff(graph_ptr))]
    floats = [offs.reshape(-1), glo.reshape(-1), gh.reshape(-1)]
    ti = torch.as_tensor(np.concatenate(ints).astype(np.int32), device=dev)
    tf = torch.as_tensor(np.concatenate(floats).astype(F32), device=dev)
    tensors = (ti, tf) + tuple(torch.split(ti, [len(a) for a in ints])) + tuple(torch.split(tf, [len(a) for a in floats]))
    out = (tensors, shifts_np, sptr, nb, len(offs))
    _PLAN_TABLES[key] = out
    while len(_PLAN_TABLES) > 16:
        _PLAN_TABLES.popitem(last=False)
    return out


def coordinate_bounds(pos: torch.Tensor) -> torch.Tensor:
    """Minimum (row 0) and maximum (row 1) of the coordinates of one graph, [2, 3] (NaN where a coordinate is)."""
    pos = pos.detach().float().contiguous()
    out = torch.empty(2, 3, dtype=torch.float32, device=pos.device)
    part = torch.empty(256, 6, dtype=torch.float32, device=pos.device)
    _lib.call("e2v2_bounds", _vp(pos), _lib.i32(pos.shape[0]), _vp(part), _vp(out), _lib.stream(pos.device))
    return out


def make_plan(pos: torch.Tensor, graph_ptr, cells, pbcs, rc: float, rmin: float = 1e-4,
              cells_per_direction: int = 4, grid_box=None, workspace: bool = True,
              src_include: Optional[torch.Tensor] = None):
    """The e2v2_nbr_plan of a batch (pos [N,3] fp32 on the GPU, graphs contiguous;
    graph_ptr, cells, pbcs on the host): per-graph shift tables, bin grids and,
    with ``workspace``, the bin workspace tensors.  Returns (plan, tensors kept
    alive for it, the shift table, its per-graph row pointers).  Without
    ``grid_box`` the atoms' bounding boxes are read back (one host sync).
    ``src_include`` ([N] bool on the GPU, or None) restricts the edge sources
    (neighbour atoms j) to the marked atoms."""
    dev = pos.device
    graph_ptr = np.asarray(graph_ptr, np.int64)
    cells = np.asarray(cells, F32).reshape(-1, 3, 3)
    pbcs = np.asarray(pbcs, bool).reshape(-1, 3)
    N = int(pos.shape[0])
    B = len(graph_ptr) - 1
    i32 = dict(dtype=torch.int32, device=dev)
    # per-graph bounding boxes (one host sync unless the caller supplies the grid box)
    if grid_box is not None:
        bb = np.asarray(grid_box, F32).reshape(2, B, 3)
    elif N:
        if B == 1 and pos.is_cuda and pos.dtype == torch.float32:
            bb = coordinate_bounds(pos).cpu().numpy().reshape(2, 1, 3)
        elif B == 1:
            bb = torch.stack([pos.amin(0, keepdim=True), pos.amax(0, keepdim=True)]).cpu().numpy()
        else:
            counts = torch.as_tensor(np.diff(graph_ptr), device=dev)
            lo = torch.segment_reduce(pos, "min", lengths=counts, axis=0, unsafe=True)
            hi = torch.segment_reduce(pos, "max", lengths=counts, axis=0, unsafe=True)
            bb = torch.stack([lo, hi]).cpu().numpy()
    else:
        bb = np.zeros((2, B, 3), F32)
    tabs = _plan_tables(dev, graph_ptr, cells, pbcs, rc, cells_per_direction, bb)
    (ti, tf, t_gptr, t_sptr, t_per, t_dim, t_base, atom_graph, t_off, t_lo, t_h), shifts_np, sptr, nb, n_off = tabs
    keep = dict(pos=pos, ti=ti, tf=tf)
    ws = [None] * 5
    if workspace:
        keep.update(atom_bin=torch.empty(max(N, 1), **i32), bin_count=torch.empty(nb, **i32),
                    bin_start=torch.empty(nb + 1, **i32), bin_atoms=torch.empty(max(N, 1), **i32),
                    stats=torch.zeros(4, **i32))
        ws = [keep[k].data_ptr() for k in ("atom_bin", "bin_count", "bin_start", "bin_atoms", "stats")]
    inc = None
    if src_include is not None:
        if src_include.shape != (N,) or src_include.device != dev:
            raise ValueError(f"src_include must be a [{N}] tensor on {dev}")
        keep["src_include"] = src_include.to(torch.uint8).contiguous()
        inc = keep["src_include"].data_ptr() if N else None
    plan = _lib.NbrPlan(N, B, nb, n_off, rc, rmin, pos.data_ptr(), atom_graph.data_ptr(), t_gptr.data_ptr(),
                        t_sptr.data_ptr(), t_per.data_ptr(), t_off.data_ptr(), t_lo.data_ptr(), t_h.data_ptr(),
                        t_dim.data_ptr(), t_base.data_ptr(), *ws, inc)
    return plan, keep, shifts_np, sptr


def build_neighbors(pos: torch.Tensor, graph_ptr, cells, pbcs, rc: float, rmin: float = 1e-4,
                    max_neighbors: Optional[int] = None, cells_per_direction: int = 4,
                    grid_box=None, src_include: Optional[torch.Tensor] = None,
                    capacity: Optional[tuple] = None, stats_host: Optional[torch.Tensor] = None) -> NeighborList:
    """pos [N,3] fp32 on the GPU (graphs contiguous); graph_ptr [B+1], cells
    [B,3,3], pbcs [B,3] on the host.  grid_box [2,B,3] (optional, host): per-graph
    (lo, hi) corners of the bin grid that contain every atom, e.g. the cell of
    positions wrapped into it; without it the atoms' bounding boxes are read back
    (one host sync).  The edge list does not depend on the grid.  An atom outside
    the supplied box is detected on the device (read back with the edge count)
    and the list is rebuilt with the bounding boxes.  src_include ([N] bool on
    the GPU, or None): only marked atoms are edge sources (every atom is still a
    query row).

    capacity = (edges, longest row): build into arrays of that many edge slots with
    no host readback at all (the kernels bound the edges on the device); the
    returned list carries ``stats`` = {E, longest row, atom outside the grid box,
    overflow} on the device, and the caller must check (later, asynchronously) that
    entries 2 and 3 are zero, else rebuild: the list is then truncated.  Needs a
    grid box, no max_neighbors.  stats_host (pinned int32 [4], optional): the
    caller's buffer the counters are copied into (no event is recorded: the caller
    synchronises, e.g. after replaying a captured graph); without it a buffer and
    an event are made here."""
    if not pos.is_cuda:
        raise RuntimeError("build_neighbors runs on the GPU only (pos must be a CUDA/HIP tensor)")
    dev = pos.device
    pos = pos.detach().to(torch.float32).contiguous()
    graph_ptr = np.asarray(graph_ptr, np.int64)
    cells = np.asarray(cells, F32).reshape(-1, 3, 3)
    pbcs = np.asarray(pbcs, bool).reshape(-1, 3)
    N = int(pos.shape[0])
    stream = _lib.stream(dev).value
    i32 = dict(dtype=torch.int32, device=dev)
    plan, keep, shifts_np, sptr = make_plan(pos, graph_ptr, cells, pbcs, rc, rmin, cells_per_direction, grid_box,
                                            src_include=src_include)
    stats = keep["stats"]
    _lib.call("e2v2_nbr_bin", _lib.C.byref(plan), _lib.vp(stream))
    row_count = torch.empty(max(N, 1), **i32)
    row_ptr = torch.empty(N + 1, **i32)
    _lib.call("e2v2_nbr_count", _lib.C.byref(plan), _lib.vp(row_count.data_ptr()), _lib.vp(row_ptr.data_ptr()),
              _lib.vp(stream))
    if capacity is not None:
        if grid_box is None or max_neighbors is not None or N == 0:
            raise ValueError("a capacity build needs a grid box, no max_neighbors and at least one atom")
        E, max_row = int(capacity[0]), int(capacity[1])
        _lib.call("e2v2_nbr_cap", _lib.vp(row_ptr.data_ptr()), _lib.i32(N), _lib.i64(E), _lib.i32(max_row),
                  _lib.vp(stats.data_ptr()), _lib.vp(stream))
        # the counters are final here: start their copy to the host now, not after the evaluation
        stats_event = None
        if stats_host is None:
            stats_host = torch.empty(4, dtype=torch.int32, pin_memory=True)
            stats_event = torch.cuda.Event()
        stats_host.copy_(stats, non_blocking=True)
        if stats_event is not None:
            stats_event.record(torch.cuda.current_stream(dev))
        outside = 0
    else:
        E, max_row, outside = (int(x) for x in stats[:3].cpu())
    if outside:
        if grid_box is None:
            raise RuntimeError("neighbour build: an atom lies outside its own bounding box")
        return build_neighbors(pos, graph_ptr, cells, pbcs, rc, rmin, max_neighbors, cells_per_direction,
                               src_include=src_include)
    f32t = dict(dtype=torch.float32, device=dev)
    tcol = torch.empty(max(E, 1), **i32); tsh = torch.empty(max(E, 1), **i32)
    tdv = torch.empty(max(E, 1), 3, **f32t); td = torch.empty(max(E, 1), **f32t)
    tkey = torch.empty(max(E, 1), dtype=torch.int64, device=dev)
    col = torch.empty(E, **i32); sh = torch.empty(E, **i32)
    dvec = torch.empty(E, 3, **f32t); dist = torch.empty(E, **f32t)
    _lib.call("e2v2_nbr_fill", _lib.C.byref(plan), _lib.vp(row_ptr.data_ptr()), _lib.i64(E), _lib.i32(max_row),
              _lib.vp(tcol.data_ptr()), _lib.vp(tsh.data_ptr()), _lib.vp(tdv.data_ptr()), _lib.vp(td.data_ptr()),
              _lib.vp(tkey.data_ptr()), _lib.vp(_ptr(col)), _lib.vp(_ptr(sh)), _lib.vp(_ptr(dvec)),
              _lib.vp(_ptr(dist)), _lib.vp(stream))
    del tcol, tsh, tdv, td
    if max_neighbors is not None and E > 0 and max_row > max_neighbors:
        cnt = torch.empty(max(N, 1), **i32)
        new_ptr = torch.empty(N + 1, **i32)
        _lib.call("e2v2_nbr_topk", _lib.vp(row_ptr.data_ptr()), _lib.i32(N), _lib.i32(int(max_neighbors)),
                  _lib.vp(cnt.data_ptr()), _lib.vp(new_ptr.data_ptr()), _lib.vp(stats.data_ptr()),
                  None, None, None, None, None, None, None, None, _lib.i32(0), _lib.vp(stream))
        E2, max_row = (int(x) for x in stats[:2].cpu())
        col2 = torch.empty(E2, **i32); sh2 = torch.empty(E2, **i32)
        dv2 = torch.empty(E2, 3, **f32t); d2 = torch.empty(E2, **f32t)
        _lib.call("e2v2_nbr_topk", _lib.vp(row_ptr.data_ptr()), _lib.i32(N), _lib.i32(int(max_neighbors)),
                  _lib.vp(cnt.data_ptr()), _lib.vp(new_ptr.data_ptr()), _lib.vp(stats.data_ptr()),
                  _lib.vp(_ptr(col)), _lib.vp(_ptr(sh)), _lib.vp(_ptr(dvec)), _lib.vp(_ptr(dist)),
                  _lib.vp(_ptr(col2)), _lib.vp(_ptr(sh2)), _lib.vp(_ptr(dv2)), _lib.vp(_ptr(d2)),
                  _lib.i32(1), _lib.vp(stream))
        row_ptr, col, sh, dvec, dist, E = new_ptr, col2, sh2, dv2, d2, E2
    edge_row = torch.empty(E, **i32)
    key_cnt = torch.empty(max(N, 1), **i32)
    key_ptr = torch.empty(N + 1, **i32)
    tstats = torch.empty(2, **i32)        # the key scan's {E, longest column} (informational)
    _lib.call("e2v2_csr_transpose", _lib.vp(row_ptr.data_ptr()), _lib.vp(_ptr(col)), _lib.i32(N), _lib.i32(N),
              _lib.i64(E), _lib.vp(_ptr(edge_row)), _lib.vp(key_cnt.data_ptr()), _lib.vp(key_ptr.data_ptr()),
              _lib.vp(tstats.data_ptr()), None, None, _lib.i32(0), _lib.vp(stream))
    key_eid = torch.empty(E, **i32)
    _lib.call("e2v2_csr_transpose", _lib.vp(row_ptr.data_ptr()), _lib.vp(_ptr(col)), _lib.i32(N), _lib.i32(N),
              _lib.i64(E), _lib.vp(_ptr(edge_row)), _lib.vp(key_cnt.data_ptr()), _lib.vp(key_ptr.data_ptr()),
              _lib.vp(tstats.data_ptr()), _lib.vp(tkey.data_ptr()), _lib.vp(_ptr(key_eid)), _lib.i32(1),
              _lib.vp(stream))
    nl = NeighborList(N, E, row_ptr, col, sh, torch.as_tensor(shifts_np), dvec, dist, edge_row, key_ptr, key_eid,
                      max_row, shift_ptr=np.asarray(sptr, np.int64))
    if capacity is not None:
        nl.stats, nl.stats_host, nl.stats_event = stats, stats_host, stats_event
    if N > 0 and E > 0:
        nl.col_span = COL_SPAN
        nl.col_slot_member, nl.col_slot_edge, nl.col_n_slots = cluster_slots(key_ptr, N, edge_row, key_eid,
                                                                             COL_SPAN)
    return nl


COL_SPAN = 4


def cluster_slots(seg_ptr: torch.Tensor, n_seg: int, member: torch.Tensor, item_eid: Optional[torch.Tensor],
                  span: int):
    """Slots of clusters of ``span`` consecutive CSR segments (e2v2_cluster_slots):
    (slot_member [items], slot_edge [items, span], n_slots [clusters])."""
    dev = seg_ptr.device
    n_items = int(member.shape[0])
    i32 = dict(dtype=torch.int32, device=dev)
    sm = torch.empty(max(n_items, 1), **i32)
    se = torch.empty(max(n_items, 1), span, **i32)
    ns = torch.empty(max((n_seg + span - 1) // span, 1), **i32)
    _lib.call("e2v2_cluster_slots", _lib.vp(seg_ptr.data_ptr()), _lib.i32(n_seg), _lib.vp(member.data_ptr()),
              _lib.vp(_ptr(item_eid)), _lib.i32(span), _lib.vp(sm.data_ptr()), _lib.vp(se.data_ptr()),
              _lib.vp(ns.data_ptr()), _lib.stream(dev))
    return sm, se, ns


def count_neighbors_noalloc(pos: torch.Tensor, graph_ptr, cells, pbcs, rc: float, rmin: float = 1e-4,
                            cells_per_direction: int = 4, grid_box=None):
    """Neighbour counts of every row through e2v2_nbr_count_noalloc (the library's
    static bin scratch instead of workspace buffers): (row_count [N], row_ptr [N+1],
    stats [3] = E, max row, outside flag), all int32 on the device.  The outputs and
    the plan's small tables are allocated here; the library call allocates nothing."""
    if not pos.is_cuda:
        raise RuntimeError("count_neighbors_noalloc runs on the GPU only")
    pos = pos.detach().to(torch.float32).contiguous()
    plan, keep, _, _ = make_plan(pos, graph_ptr, cells, pbcs, rc, rmin, cells_per_direction, grid_box,
                                 workspace=False)
    N = int(pos.shape[0])
    i32 = dict(dtype=torch.int32, device=pos.device)
    row_count = torch.empty(max(N, 1), **i32)
    row_ptr = torch.empty(N + 1, **i32)
    stats = torch.empty(3, **i32)
    _lib.call("e2v2_nbr_count_noalloc", _lib.C.byref(plan), _lib.vp(row_count.data_ptr()),
              _lib.vp(row_ptr.data_ptr()), _lib.vp(stats.data_ptr()),
              _lib.stream(pos.device))
    return row_count[:N], row_ptr, stats


def construct_radius_neighbor(node_pos, node_mask, expand_node_pos, expand_node_mask, max_dist, include_mask=None,
                              min_dist=-1, max_neighbors=None, error_check=False, poly="poly", toy_config=None):
    """The reference's padded-batch neighbour search with its signature and
    output dict (module_utils.py:3119-3242), on the HIP pair kernels.

    node_pos [B, L, 3], node_mask [B, L] (True = atom), expand_node_pos
    [B, L2, 3], expand_node_mask [B, L2], include_mask [B, L2] or None.  Query
    q is the q-th real atom (node_pos[node_mask]); it meets every padded
    expanded position of its batch row (padding included, as in the
    reference, whose callers place padding at 999 A).  Pairs with
    min_dist <= d <= max_dist (and included) are kept, each row sorted by
    (d, expanded slot) and cut to topK = max(min(L2, max_neighbors, longest
    row), 1).  Returns query_idx, neighbor_idx (int64, the index into
    expand_node_pos[expand_node_mask], clamped to its last row), metadata
    (the 6-tuple of prepare_sparse_qk_edge_index_metadata), f_edge_vec
    (node_pos[q] - the indexed expanded node), f_dist, f_poly_dist
    (polynomial(d, max_dist), or smooth_polynomial_bell(d, min_dist, max_dist)
    for poly="poly_bell").  Positions are evaluated in fp32 with d =
    sqrt((dx dx + dy dy) + dz dz).  toy_config {"prob": p} drops each kept
    edge with probability p (the reference's random attention mask, drawn per
    edge here).  A batch with no real atom raises, as the reference's max over
    an empty selection does."""
    from .sparse_ops import prepare_sparse_qk_edge_index_metadata
    import logging

    if poly not in ("poly", "poly_bell"):
        raise ValueError("sorry, you must set poly or poly_bell")
    for t in (node_pos, expand_node_pos):
        if not t.is_cuda:
            raise RuntimeError("construct_radius_neighbor runs on the GPU only (HIP library, no CPU path)")
    dev = node_pos.device
    B, L = node_pos.shape[:2]
    L2 = expand_node_pos.shape[1]
    node_mask = node_mask.to(torch.bool)
    expand_node_mask = expand_node_mask.to(torch.bool)
    if tuple(node_mask.shape) != (B, L) or tuple(expand_node_mask.shape) != (B, L2) \
            or expand_node_pos.shape[0] != B:
        raise ValueError(f"shapes: node_pos {tuple(node_pos.shape)}, node_mask {tuple(node_mask.shape)}, "
                         f"expand_node_pos {tuple(expand_node_pos.shape)}, "
                         f"expand_node_mask {tuple(expand_node_mask.shape)}")
    pos32 = node_pos.detach().to(torch.float32)
    qpos = pos32[node_mask].contiguous()
    qgraph = node_mask.nonzero()[:, 0].to(torch.int32).contiguous()
    N = qpos.shape[0]
    if N == 0:
        raise RuntimeError("construct_radius_neighbor: node_mask selects no atom")
    spos = expand_node_pos.detach().to(torch.float32).contiguous()
    sflat = spos[expand_node_mask].contiguous()
    n_flat = sflat.shape[0]
    expand_ptr = torch.zeros(B + 1, dtype=torch.int64, device=dev)
    expand_ptr[1:] = torch.cumsum(expand_node_mask.sum(-1), 0)
    sbase = expand_ptr[:B].to(torch.int32).contiguous()
    inc = None
    if include_mask is not None:
        inc = include_mask.to(torch.bool).reshape(B, L2).to(torch.uint8).contiguous()
    plan = _lib.PairPlan(N, B, L2, n_flat, float(max_dist), float(min_dist), 0 if poly == "poly" else 1,
                         _vp(qpos), _vp(qgraph), _vp(spos), _vp(inc), _vp(sbase), _vp(sflat))
    stream = _lib.stream(dev)
    i32 = dict(dtype=torch.int32, device=dev)
    row_count = torch.empty(N, **i32)
    row_ptr = torch.empty(N + 1, **i32)
    stats = torch.zeros(3, **i32)
    _lib.call("e2v2_pair_count", _lib.C.byref(plan), _vp(row_count), _vp(row_ptr), _vp(stats), stream)
    n_pairs, longest = (int(x) for x in stats[:2].cpu())
    top_k = max(min(L2, longest) if max_neighbors is None else min(L2, int(max_neighbors), longest), 1)
    new_ptr, E = row_ptr, n_pairs
    if top_k < longest:
        cnt = torch.empty(N, **i32)
        new_ptr = torch.empty(N + 1, **i32)
        _lib.call("e2v2_nbr_topk", _vp(row_ptr), _lib.i32(N), _lib.i32(top_k), _vp(cnt), _vp(new_ptr),
                  _vp(stats), None, None, None, None, None, None, None, None, _lib.i32(0), stream)
        E = int(stats[0].item())
    query_idx = torch.empty(E, dtype=torch.int64, device=dev)
    neighbor_idx = torch.empty(E, dtype=torch.int64, device=dev)
    f_edge_vec = torch.empty(E, 3, dtype=torch.float32, device=dev)
    f_dist = torch.empty(E, dtype=torch.float32, device=dev)
    f_poly = torch.empty(E, dtype=torch.float32, device=dev)
    if E > 0:
        tkey = torch.empty(n_pairs, dtype=torch.int64, device=dev)
        _lib.call("e2v2_pair_emit", _lib.C.byref(plan), _vp(row_ptr), _lib.i64(n_pairs), _lib.i32(longest),
                  _vp(new_ptr), _vp(tkey), _vp(query_idx), _vp(neighbor_idx), _vp(f_edge_vec), _vp(f_dist),
                  _vp(f_poly), stream)
    if toy_config is not None and E > 0:
        keep = torch.rand(E, device=dev) >= float(toy_config.get("prob", 0))
        query_idx, neighbor_idx = query_idx[keep].contiguous(), neighbor_idx[keep].contiguous()
        f_edge_vec, f_dist, f_poly = f_edge_vec[keep].contiguous(), f_dist[keep].contiguous(), f_poly[keep].contiguous()
    if error_check:
        log = logging.getLogger(__name__)
        if f_dist.numel() and torch.max(torch.linalg.norm(f_edge_vec, dim=-1) - f_dist) != 0:
            log.error("Please verify your code, neighbor selection error happened")
        if torch.sum(node_pos[~node_mask] == 0):
            log.warning("node padding part is zero, will lead to some neighbor dist sort error")
        if torch.sum(expand_node_pos[~expand_node_mask] == 0):
            log.warning("expand_node_pos padding part is zero, will lead to some neighbor dist sort error")
    return {
        "query_idx": query_idx,
        "neighbor_idx": neighbor_idx,
        "metadata": prepare_sparse_qk_edge_index_metadata(query_idx, neighbor_idx, N, n_flat),
        "f_edge_vec": f_edge_vec,
        "f_dist": f_dist,
        "f_poly_dist": f_poly,
    }


def neighbor_list_from_edges(row_ptr: torch.Tensor, src_atom: torch.Tensor, dvec: torch.Tensor, dist: torch.Tensor,
                             n_atoms: int, clusters: bool = True) -> NeighborList:
    """A NeighborList over an edge list already in query-row order (row_ptr
    [n_atoms + 1] int32, the source atom of every edge, its dvec [E,3] and
    dist [E]), for callers that bring their own edges (the reference's
    construct_radius_neighbor dict): key CSR by source atom (edges of each
    column in edge order) and the column clusters of the attention backward
    built on the GPU.  Shifts are not tracked (shift_idx zero)."""
    dev = dvec.device
    N = int(n_atoms)
    E = int(src_atom.shape[0])
    i32 = dict(dtype=torch.int32, device=dev)
    row_ptr = row_ptr.to(torch.int32).contiguous()
    col = src_atom.to(torch.int32).contiguous()
    dvec = dvec.detach().to(torch.float32).contiguous()
    dist = dist.detach().to(torch.float32).contiguous()
    if row_ptr.numel() != N + 1 or dvec.shape != (E, 3) or dist.shape != (E,):
        raise ValueError(f"edge list shapes: row_ptr {tuple(row_ptr.shape)} for {N} atoms, dvec {tuple(dvec.shape)}, "
                         f"dist {tuple(dist.shape)}, {E} edges")
    if E > 0:   # the CSR kernels index with these: one host read to check them
        lo, hi, p0, pe, bad = (int(x) for x in torch.stack([
            col.min(), col.max(), row_ptr[0], row_ptr[-1], (row_ptr[1:] < row_ptr[:-1]).sum().to(torch.int32)]).cpu())
        if lo < 0 or hi >= N or p0 != 0 or pe != E or bad:
            raise ValueError(f"edge list: source atoms in [{lo}, {hi}] for {N} atoms, row_ptr from {p0} to {pe} "
                             f"for {E} edges, {bad} decreasing steps")
    stream = _lib.stream(dev)
    stats = torch.zeros(3, **i32)
    edge_row = torch.empty(E, **i32)
    key_cnt = torch.empty(max(N, 1), **i32)
    key_ptr = torch.empty(N + 1, **i32)
    key_eid = torch.empty(E, **i32)
    tkey = torch.empty(max(E, 1), dtype=torch.int64, device=dev)
    for phase in (0, 1):
        _lib.call("e2v2_csr_transpose", _vp(row_ptr), _vp(col), _lib.i32(N), _lib.i32(N), _lib.i64(E),
                  _vp(edge_row), _vp(key_cnt), _vp(key_ptr), _vp(stats), _vp(tkey) if phase else None,
                  _vp(key_eid) if phase else None, _lib.i32(phase), stream)
    nl = NeighborList(N, E, row_ptr, col, torch.zeros(E, **i32), torch.zeros(1, 3, dtype=torch.int32), dvec, dist,
                      edge_row, key_ptr, key_eid, 0)
    if clusters and N > 0 and E > 0:
        nl.col_span = COL_SPAN
        nl.col_slot_member, nl.col_slot_edge, nl.col_n_slots = cluster_slots(key_ptr, N, edge_row, key_eid,
                                                                             COL_SPAN)
    return nl
