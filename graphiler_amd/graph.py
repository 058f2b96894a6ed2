"""Graph container and host-side preparation.

``DGLGraph`` mirrors the reference's custom class
(include/dglgraph.h:7-75, registered in src/dglgraph.cpp:5-24): the same ten
constructor arguments, the same four setters and the same public fields, so the
operator wrappers in :mod:`graphiler_amd.ops` read it exactly as the
reference's operators read theirs.  On top of that it caches what the gfx950
kernels need once per graph: the slot->row maps of both adjacencies, whether
the edge-id columns are the identity, and a reusable workspace.

``prepare_graph`` mirrors python/graphiler/utils/setup.py:116-146: in- and
out-adjacency with int32 pointer / neighbour / edge-id columns and int64 COO
columns, built here from a plain (src, dst) edge list instead of a DGL graph.
Inside one node's group the edges keep ascending edge-id order.
"""
from __future__ import annotations

from dataclasses import dataclass
from typing import Optional

import numpy as np
import torch

from . import capi


@dataclass
class GraphArrays:
    """Host (numpy) form of the arrays ``prepare_graph`` produces."""
    num_nodes: int
    in_pointer: np.ndarray
    in_node_indices: np.ndarray
    in_edge_indices: np.ndarray
    out_pointer: np.ndarray
    out_node_indices: np.ndarray
    out_edge_indices: np.ndarray
    COO_src: np.ndarray
    COO_dst: np.ndarray


def _group(n_nodes: int, key: np.ndarray, other: np.ndarray):
    """Stable grouping of edge ids by ``key`` -> (pointer, neighbour, edge id)."""
    order = np.argsort(key, kind="stable")
    counts = np.bincount(key, minlength=n_nodes)
    pointer = np.zeros(n_nodes + 1, np.int64)
    np.cumsum(counts, out=pointer[1:])
    return (pointer.astype(np.int32), other[order].astype(np.int32),
            order.astype(np.int32))


def build_graph_arrays(src, dst, num_nodes: int) -> GraphArrays:
    """CSR-by-destination and CSR-by-source of an edge list (host, numpy)."""
    src = np.ascontiguousarray(src, dtype=np.int64)
    dst = np.ascontiguousarray(dst, dtype=np.int64)
    if src.shape != dst.shape or src.ndim != 1:
        raise ValueError("src and dst must be 1-D arrays of equal length")
    if src.shape[0] >= 2 ** 31 or num_nodes >= 2 ** 31:
        raise ValueError("graphs are limited to int32 node and edge ids")
    if src.size and (min(src.min(), dst.min()) < 0 or
                     max(src.max(), dst.max()) >= num_nodes):
        raise ValueError("edge endpoint outside [0, num_nodes)")
    ip, inb, ie = _group(num_nodes, dst, src)
    op, onb, oe = _group(num_nodes, src, dst)
    return GraphArrays(num_nodes, ip, inb, ie, op, onb, oe, src, dst)


def type_pointer(type_of, num_types: int) -> np.ndarray:
    """int32 running sum of items per type; ``type_of`` must be sorted
    (ids of one type are contiguous, include/dglgraph.h:68-69)."""
    type_of = np.asarray(type_of, dtype=np.int64)
    if type_of.size and np.any(np.diff(type_of) < 0):
        raise ValueError("items must be sorted by type")
    ptr = np.zeros(num_types + 1, np.int64)
    np.cumsum(np.bincount(type_of, minlength=num_types), out=ptr[1:])
    return ptr.astype(np.int32)


def sort_edges_by_type(src, dst, etype):
    """Stable reorder of an edge list so edge ids of one type are contiguous.
    Returns (src, dst, etype, order) with ``order`` the applied permutation."""
    etype = np.asarray(etype, dtype=np.int64)
    order = np.argsort(etype, kind="stable")
    return (np.asarray(src)[order], np.asarray(dst)[order], etype[order], order)


def _check_index(t: torch.Tensor, dtype: torch.dtype, name: str):
    if t.dtype != dtype:
        raise RuntimeError(f"{name} must be {dtype}")
    if not t.is_contiguous():
        raise RuntimeError(f"{name} must be contiguous")


class DGLGraph:
    """Drop-in for ``torch.classes.my_classes.DGLGraph``."""

    def __init__(self, in_pointer, in_node_indices, in_edge_indices,
                 out_pointer, out_node_indices, out_edge_indices, COO_src,
                 COO_dst, ntype_pointer: Optional[torch.Tensor] = None,
                 etype_pointer: Optional[torch.Tensor] = None):
        for name, t in (("in_pointer", in_pointer),
                        ("in_node_indices", in_node_indices),
                        ("in_edge_indices", in_edge_indices),
                        ("out_pointer", out_pointer),
                        ("out_node_indices", out_node_indices),
                        ("out_edge_indices", out_edge_indices)):
            _check_index(t, torch.int32, name)
        _check_index(COO_src, torch.int64, "COO_src")
        _check_index(COO_dst, torch.int64, "COO_dst")
        self.in_pointer = in_pointer
        self.in_node_indices = in_node_indices
        self.in_edge_indices = in_edge_indices
        self.out_pointer = out_pointer
        self.out_node_indices = out_node_indices
        self.out_edge_indices = out_edge_indices
        self.COO_src = COO_src
        self.COO_dst = COO_dst
        self.ntype_pointer = None
        self.etype_pointer = None
        self.ntype_COO = None
        self.etype_COO = None
        # include/dglgraph.h:22-27
        self.num_nodes = int(in_pointer.size(0)) - 1
        self.num_edges = int(in_node_indices.size(0))
        self.num_ntypes = 1
        self.num_etypes = 1
        self._cache = {}
        self.SetNtypePointer(ntype_pointer)
        self.SetEtypePointer(etype_pointer)

    # -- setters (include/dglgraph.h:29-46) ---------------------------------
    def SetNtypePointer(self, pointer):
        if pointer is not None:
            _check_index(pointer, torch.int32, "ntype_pointer")
        self.ntype_pointer = pointer
        self.num_ntypes = int(pointer.size(0)) - 1 if pointer is not None else 1

    def SetEtypePointer(self, pointer):
        if pointer is not None:
            _check_index(pointer, torch.int32, "etype_pointer")
        self.etype_pointer = pointer
        self.num_etypes = int(pointer.size(0)) - 1 if pointer is not None else 1
        # the layouts prepared from the edge types belong to the old pointer (a layout
        # already handed to a launch stays alive with that launch's tensors)
        self._cache.pop("typed_tiles", None)
        self._cache.pop("pairs", None)

    def SetNtypeCOO(self, column):
        _check_index(column, torch.int64, "ntype_COO")
        if column.size(0) != self.num_nodes:
            raise RuntimeError("ntype_COO must have one entry per node")
        self.ntype_COO = column

    def SetEtypeCOO(self, column):
        _check_index(column, torch.int64, "etype_COO")
        if column.size(0) != self.num_edges:
            raise RuntimeError("etype_COO must have one entry per edge")
        self.etype_COO = column

    # -- derived data the kernels schedule with -----------------------------
    @property
    def device(self):
        return self.in_pointer.device

    def _row_ids(self, pointer: torch.Tensor) -> torch.Tensor:
        rows = torch.empty(self.num_edges, dtype=torch.int32, device=self.device)
        stream = torch.cuda.current_stream(self.device).cuda_stream
        capi.check(capi.load().ga_csr_row_ids(
            pointer.data_ptr(), self.num_nodes, self.num_edges,
            rows.data_ptr(), stream), "ga_csr_row_ids")
        return rows

    def _kept_row_ids(self, key: str, pointer: torch.Tensor) -> torch.Tensor:
        rows = self._cache.get(key)
        if rows is None:
            rows = self._row_ids(pointer)
            # inside a capture nothing runs yet and the memory is the recorded graph's: that
            # graph fills its own column on every replay, the next eager call one to keep
            if not torch.cuda.is_current_stream_capturing():
                self._cache[key] = rows
        return rows

    @property
    def in_row_of_slot(self) -> torch.Tensor:
        """Destination node of every slot of the in-adjacency (int32, E)."""
        return self._kept_row_ids("in_rows", self.in_pointer)

    @property
    def out_row_of_slot(self) -> torch.Tensor:
        """Source node of every slot of the out-adjacency (int32, E)."""
        return self._kept_row_ids("out_rows", self.out_pointer)

    def _identity(self, key: str, column: torch.Tensor) -> bool:
        if key not in self._cache:
            n = column.numel()
            ar = torch.arange(n, dtype=torch.int32, device=column.device)
            self._cache[key] = bool(torch.equal(column, ar))
        return self._cache[key]

    @property
    def max_in_degree(self) -> int:
        """Largest number of in-edges of a node (one reduction and host read, then cached)."""
        if "max_in_degree" not in self._cache:
            self._cache["max_in_degree"] = int(torch.diff(self.in_pointer).max().item()) \
                if self.num_nodes > 0 else 0
        return self._cache["max_in_degree"]

    @property
    def in_eid_is_identity(self) -> bool:
        """True when edge ids already are in-adjacency slot numbers."""
        return self._identity("in_ident", self.in_edge_indices)

    @property
    def out_eid_is_identity(self) -> bool:
        return self._identity("out_ident", self.out_edge_indices)

    def relation_pairs(self) -> Optional["RelationPairs"]:
        """The (destination, relation) pairs of the in-adjacency, built once on the
        device: a layer whose per-edge work is linear in a per-relation matrix (HGT's
        ``bmm(k, relation_att)`` and ``bmm(v, relation_msg)``, examples/HGT/HGT.py:35-44)
        can apply that matrix once per pair instead of once per edge.  None when the
        graph has no edge types or the slots of a destination are not grouped by
        relation (they are when edge ids are sorted by type, as
        include/dglgraph.h:24-27 requires for the type pointer)."""
        if "pairs" not in self._cache:
            self._cache["pairs"] = _build_relation_pairs(self)
        return self._cache["pairs"]

    def _source_degrees(self):
        """(nodes, edges) by the power of two below the out-degree, as host int64 arrays."""
        if "source_degrees" not in self._cache:
            both = torch.empty((2, capi.GA_DEGREE_BUCKETS), dtype=torch.int64, device=self.device)
            capi.check(capi.load().ga_degree_buckets(
                self.out_pointer.data_ptr(), self.num_nodes, both.data_ptr(),
                torch.cuda.current_stream(self.device).cuda_stream), "ga_degree_buckets")
            self._cache["source_degrees"] = both.cpu().numpy()
        return self._cache["source_degrees"]

    def source_classes(self, feat: int, dtype: int) -> Optional["SourceClasses"]:
        """The slots of the in-adjacency ordered by classes of their sources, where a sum
        of rows of ``feat`` features is faster over them (``ga_spmm_source_classes``),
        else None.  Degrees are read and a layout is built on first use, neither while the
        stream is captured; a layout that does not fit the memory is done without."""
        lib = capi.load()
        key = ("source_classes", feat, dtype)
        n = self._cache.get(key)
        if n is None:
            if not lib.ga_spmm_source_classes(None, None, self.num_nodes, self.num_edges, feat, dtype):
                n = 0
            elif torch.cuda.is_current_stream_capturing():
                return None
            else:
                nodes, edges = self._source_degrees()
                n = int(lib.ga_spmm_source_classes(nodes.ctypes.data, edges.ctypes.data,
                                                   self.num_nodes, self.num_edges, feat, dtype))
            self._cache[key] = n
        if n == 0:
            return None
        layout = self._cache.get(("classes", n))
        if layout is None:
            if torch.cuda.is_current_stream_capturing():
                return None
            try:
                layout = _build_source_classes(self, n)
            except torch.OutOfMemoryError:
                self._cache[key] = 0
                return None
            self._cache[("classes", n)] = layout
        return layout

    def rows_by_length(self) -> Optional["RowsByLength"]:
        """The order in which a GAT layer over its inputs walks the destinations: built on the
        device at first use and kept with the graph; None where that would have to happen while a
        stream is captured, or does not fit the memory now."""
        rows = self._cache.get("rows_by_length")
        if rows is None:
            if torch.cuda.is_current_stream_capturing():
                return None
            try:
                rows = self._cache["rows_by_length"] = _build_rows_by_length(self)
            except torch.OutOfMemoryError:
                return None
        return rows

    def refuse_source_classes(self, feat: int, dtype: int) -> None:
        """The scratch of ``feat`` features over source classes does not fit: the plain sum
        from now on.  A layout that no launch has read is given back; one that has been
        read stays, a recorded HIP graph may replay launches over it."""
        n, self._cache[("source_classes", feat, dtype)] = self._cache[("source_classes", feat, dtype)], 0
        if not self._cache[("classes", n)].used:
            del self._cache[("classes", n)]

    def workspace(self, nbytes: int) -> torch.Tensor:
        """Scratch buffer shared by the operators called on this graph (grows on
        demand).  Calls that use it must be ordered on one stream: two streams
        working on one graph object race on it.  A buffer that was handed out is
        kept alive as long as the graph, because a recorded HIP graph may still
        replay launches that write to it."""
        ws = self._cache.get("ws")
        if ws is None or ws.numel() < nbytes:
            larger = torch.empty(max(int(nbytes), 256), dtype=torch.uint8,
                                 device=self.device)
            if ws is not None:
                self._cache.setdefault("retired_ws", []).append(ws)
            self._cache["ws"] = ws = larger
        return ws


@dataclass
class RelationPairs:
    """Slots of the in-adjacency grouped into runs of one (destination, relation).
    Pairs are numbered in slot order (by destination, then relation); ``by_type``
    lists them by relation (stable), which is the row order the typed products need."""
    num_pairs: int
    max_slots: int                  # slots of the largest pair
    pair_pointer: torch.Tensor      # (P + 1) int32: first slot of every pair
    pair_of_slot: torch.Tensor      # (E) int32
    pair_dst: torch.Tensor          # (P) int32, ascending
    dst_pointer: torch.Tensor       # (N + 1) int32: first pair of every destination
    type_pointer: torch.Tensor      # (T + 1) int32 over by_type
    by_type: torch.Tensor           # (P) int64: pair ids ordered by relation
    rank: torch.Tensor              # (P) int32: position of a pair in by_type
    rank_of_slot: torch.Tensor      # (E) int32: rank[pair_of_slot]
    dst_by_type: torch.Tensor       # (P) int64: pair_dst[by_type]
    rows: torch.Tensor              # (P, 4) int32 in by_type order: first slot, end slot, destination, 0
    tiles: torch.Tensor             # (-, 4) int32: type (-1: none), first row, end row, 0


def _build_relation_pairs(g: "DGLGraph") -> Optional[RelationPairs]:
    if g.etype_pointer is None or g.num_edges == 0:
        return None
    dev, n_edges, n_types = g.device, g.num_edges, g.num_etypes
    rows = g.in_row_of_slot.long()
    eid = g.in_edge_indices.long()
    etype = torch.bucketize(eid, g.etype_pointer[1:].long(), right=True)
    key = rows * n_types + etype
    if n_edges > 1 and not bool((key[1:] >= key[:-1]).all()):
        return None
    first = torch.ones(n_edges, dtype=torch.bool, device=dev)
    first[1:] = key[1:] != key[:-1]
    pair_of_slot = torch.cumsum(first, 0) - 1
    starts = torch.nonzero(first).reshape(-1)
    n_pairs = int(starts.numel())
    pair_key = key[starts]
    pair_dst = torch.div(pair_key, n_types, rounding_mode="floor")
    pair_type = pair_key - pair_dst * n_types
    by_type = torch.argsort(pair_type, stable=True)
    rank = torch.empty_like(by_type).scatter_(0, by_type, torch.arange(n_pairs, device=dev))
    bounds = torch.cat([starts, starts.new_full((1,), n_edges)])
    largest = torch.diff(bounds).max()
    pairs = RelationPairs(
        num_pairs=n_pairs,
        max_slots=0,
        pair_pointer=bounds.int().contiguous(),
        pair_of_slot=pair_of_slot.int().contiguous(),
        pair_dst=pair_dst.int().contiguous(),
        dst_pointer=torch.searchsorted(pair_dst.contiguous(),
                                       torch.arange(g.num_nodes + 1, device=dev)).int().contiguous(),
        type_pointer=torch.searchsorted(pair_type[by_type].contiguous(),
                                        torch.arange(n_types + 1, device=dev)).int().contiguous(),
        by_type=by_type.contiguous(),
        rank=rank.int().contiguous(),
        rank_of_slot=rank[pair_of_slot].int().contiguous(),
        dst_by_type=pair_dst[by_type].contiguous(),
        rows=torch.empty((n_pairs, 4), dtype=torch.int32, device=dev),
        tiles=torch.empty((int(capi.load().ga_pair_tiles_capacity(n_pairs, n_types)), 4),
                          dtype=torch.int32, device=dev))
    capi.check(capi.load().ga_pair_tiles_build(
        pairs.type_pointer.data_ptr(), n_types, pairs.by_type.data_ptr(),
        pairs.dst_by_type.data_ptr(), pairs.pair_pointer.data_ptr(), n_pairs, pairs.rows.data_ptr(),
        pairs.tiles.data_ptr(), torch.cuda.current_stream(dev).cuda_stream), "ga_pair_tiles_build")
    pairs.max_slots = int(largest.item())      # read behind all launches: the host waits once
    return pairs


@dataclass
class RowsByLength:
    """Destinations ordered by their number of in-edges, long ones cut into pieces."""
    rows: torch.Tensor              # (N, 4) int32: node, first slot, end slot, 0
    n_light: int                    # rows of at most `longest` slots, in front
    n_pieces: int                   # capacity of `pieces`
    piece_first: torch.Tensor       # (long rows + 1) int32
    pieces: torch.Tensor            # (n_pieces, 2) int32: first and end slot


def _build_rows_by_length(g: "DGLGraph") -> RowsByLength:
    lib, dev, n = capi.load(), g.device, g.num_nodes
    current = torch.cuda.current_stream(dev)
    stream = current.cuda_stream
    i32 = dict(dtype=torch.int32, device=dev)
    longest = int(lib.ga_gat_rows_longest(g.num_edges))
    rows, light = torch.empty((n, 4), **i32), torch.empty(1, **i32)
    ws = torch.empty(int(lib.ga_gat_rows_workspace_bytes(n, longest)), dtype=torch.uint8, device=dev)
    capi.check(lib.ga_gat_rows_build(g.in_pointer.data_ptr(), n, longest, rows.data_ptr(), light.data_ptr(),
                                     ws.data_ptr(), ws.numel(), stream), "ga_gat_rows_build")
    n_light = int(light.item())
    n_long = n - n_light
    n_pieces = g.num_edges // longest + n_long if n_long else 0
    out = RowsByLength(rows, n_light, n_pieces, torch.empty(n_long + 1, **i32),
                       torch.empty((max(n_pieces, 1), 2), **i32))
    if n_long:
        capi.check(lib.ga_gat_pieces_build(rows[n_light:].data_ptr(), n_long, longest,
                                           out.piece_first.data_ptr(), out.pieces.data_ptr(), stream),
                   "ga_gat_pieces_build")
        current.synchronize()       # the next call may come on another stream, which waits for nothing
    return out


@dataclass
class SourceClasses:
    """Slots of the in-adjacency ordered by (class of the source, destination)."""
    num_classes: int
    pointer: torch.Tensor           # (classes * N + 1) int32
    rows: torch.Tensor              # (E) int32: class * N + destination
    nbr: torch.Tensor               # (E) int32: source
    used: bool = False              # a launch has read it


def _build_source_classes(g: "DGLGraph", n: int) -> SourceClasses:
    lib = capi.load()
    i32 = dict(dtype=torch.int32, device=g.device)
    out = SourceClasses(n, torch.empty(n * g.num_nodes + 1, **i32),
                        torch.empty(g.num_edges, **i32), torch.empty(g.num_edges, **i32))
    ws = torch.empty(int(lib.ga_source_classes_workspace_bytes(g.num_edges, n)),
                     dtype=torch.uint8, device=g.device)
    capi.check(lib.ga_source_classes_build(
        g.in_row_of_slot.data_ptr(), g.in_node_indices.data_ptr(), g.num_nodes, g.num_edges, n,
        out.pointer.data_ptr(), out.rows.data_ptr(), out.nbr.data_ptr(), ws.data_ptr(),
        ws.numel(), torch.cuda.current_stream(g.device).cuda_stream), "ga_source_classes_build")
    return out


def group_on_device(key: torch.Tensor, other: Optional[torch.Tensor], n_keys: int):
    """Stable grouping of item ids by ``key`` on the GPU (setup.py:116-146):
    returns (pointer int32 (n_keys+1), other[order] int32 or None, order int32,
    status int32 (1,)).  ``status`` is left on the device: 1 means a key outside
    [0, n_keys); read it when convenient."""
    from . import capi
    if key.dtype != torch.int64 or not key.is_cuda or not key.is_contiguous():
        raise RuntimeError("key must be a contiguous int64 CUDA tensor")
    if other is not None and (other.dtype != torch.int64 or other.shape != key.shape
                              or not other.is_cuda or not other.is_contiguous()):
        raise RuntimeError("other must match key (contiguous int64 CUDA tensor)")
    n, dev = int(key.numel()), key.device
    if n >= 2 ** 31 or n_keys >= 2 ** 31 - 1:
        raise ValueError("graphs are limited to int32 node and edge ids")
    lib = capi.load()
    pointer = torch.empty(n_keys + 1, dtype=torch.int32, device=dev)
    order = torch.empty(n, dtype=torch.int32, device=dev)
    nbr = torch.empty(n, dtype=torch.int32, device=dev) if other is not None else None
    status = torch.empty(1, dtype=torch.int32, device=dev)
    ws = torch.empty(max(int(lib.ga_group_edges_workspace_bytes(n_keys, n)), 256),
                     dtype=torch.uint8, device=dev)
    capi.check(lib.ga_group_edges(
        key.data_ptr(), None if other is None else other.data_ptr(), n_keys, n,
        pointer.data_ptr(), None if nbr is None else nbr.data_ptr(), order.data_ptr(),
        status.data_ptr(), ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream(dev).cuda_stream), "ga_group_edges")
    return pointer, nbr, order, status


def _group_both(src: torch.Tensor, dst: torch.Tensor, num_nodes: int, status: torch.Tensor):
    """Both adjacencies of an edge list: group_on_device(dst, src) and
    group_on_device(src, dst) in the same launches; ``status`` int32 (2,): a dst, a src
    outside [0, num_nodes)."""
    n, dev = int(src.numel()), src.device
    lib = capi.load()
    i32 = dict(dtype=torch.int32, device=dev)
    sides = [(torch.empty(num_nodes + 1, **i32), torch.empty(n, **i32), torch.empty(n, **i32))
             for _ in range(2)]
    ws = torch.empty(max(int(lib.ga_group_edges_both_workspace_bytes(num_nodes, n)), 256),
                     dtype=torch.uint8, device=dev)
    capi.check(lib.ga_group_edges_both(
        src.data_ptr(), dst.data_ptr(), num_nodes, n, *(t.data_ptr() for side in sides for t in side),
        status.data_ptr(), ws.data_ptr(), ws.numel(),
        torch.cuda.current_stream(dev).cuda_stream), "ga_group_edges_both")
    return sides


# Host columns go to the device as 32-bit ids, which is all that a valid one holds, and are
# widened there: the link moves half the bytes.  Pieces of this many ids go through page-locked
# memory, narrowed and checked by all host threads while the piece before is on its way (82 us
# for a full one).  The host's calls per piece bound small columns: 17 MB of edges and types in
# pieces of 2 MB 330 us, of 4 MB 263, as 64-bit ids 460.  A column below a sixteenth of a piece
# goes over directly.
_UPLOAD_PIECE = 1 << 20
_UPLOAD_PIECES = 3


def _upload(arrays, dev):
    """int64 host arrays as device tensors, on the current stream.  The pieces come from
    torch's host allocator and are given back on return; one is written again only when
    the copy out of it is done."""
    outs = [torch.empty(a.shape, dtype=torch.int64, device=dev) for a in arrays]
    ring, used = [], 0
    for a, out in zip(arrays, outs):
        host, out = torch.from_numpy(a).view(-1), out.view(-1)
        if a.size < _UPLOAD_PIECE // 16:
            out.copy_(host)
            continue
        narrow = torch.empty(a.size, dtype=torch.int32, device=dev)
        for lo in range(0, a.size, _UPLOAD_PIECE):
            n = min(_UPLOAD_PIECE, a.size - lo)
            if len(ring) < _UPLOAD_PIECES:
                ring.append((torch.empty(_UPLOAD_PIECE, dtype=torch.int32, pin_memory=True),
                             torch.cuda.Event()))
            piece, done = ring[used % _UPLOAD_PIECES]
            if used >= _UPLOAD_PIECES:
                done.synchronize()
            piece[:n].copy_(host[lo:lo + n])
            narrow[lo:lo + n].copy_(piece[:n], non_blocking=True)
            done.record(torch.cuda.current_stream(dev))
            used += 1
            least, most = torch.aminmax(host[lo:lo + n])
            if int(least) < -2 ** 31 or int(most) >= 2 ** 31:
                out.copy_(host)         # no id of a graph: whole, for whoever reports it
                break
        else:
            out.copy_(narrow)
    return outs


def _sorted_pointer(key: torch.Tensor, n_keys: int, status: Optional[torch.Tensor] = None):
    """(pointer int32 (n_keys + 1), status int32 (2,)) of sorted keys; the status (a key
    outside [0, n_keys), a key below its predecessor) is left on the device."""
    n, dev = int(key.numel()), key.device
    if n >= 2 ** 31 or n_keys >= 2 ** 31 - 1:
        raise ValueError("graphs are limited to int32 node and edge ids")
    pointer = torch.empty(n_keys + 1, dtype=torch.int32, device=dev)
    if status is None:
        status = torch.empty(2, dtype=torch.int32, device=dev)
    capi.check(capi.load().ga_sorted_pointer(
        key.data_ptr(), n_keys, n, pointer.data_ptr(), status.data_ptr(),
        torch.cuda.current_stream(dev).cuda_stream), "ga_sorted_pointer")
    return pointer, status


def prepare_graph(src, dst, num_nodes: int, device="cuda:0",
                  ntype_of=None, num_ntypes: int = 0, etype_of=None,
                  num_etypes: int = 0) -> DGLGraph:
    """Build the device graph from an edge list (setup.py:116-146); when type
    columns are given also install the type pointers and type COO columns the
    way load_data does for heterogeneous graphs (setup.py:87-100).  The edge
    list is uploaded once and grouped on the GPU (both adjacencies and the type
    pointers); nothing is sorted on the host."""
    dev = torch.device(device)
    src = np.ascontiguousarray(src, dtype=np.int64)
    dst = np.ascontiguousarray(dst, dtype=np.int64)
    if src.shape != dst.shape or src.ndim != 1:
        raise ValueError("src and dst must be 1-D arrays of equal length")
    if src.shape[0] >= 2 ** 31 or num_nodes >= 2 ** 31 - 1:
        raise ValueError("graphs are limited to int32 node and edge ids")
    given = [None if t is None else np.ascontiguousarray(t, dtype=np.int64)
             for t in (ntype_of, etype_of)]
    with torch.cuda.device(dev):
        up = _upload([src, dst] + [t for t in given if t is not None], dev)
        coo_src, coo_dst, types = up[0], up[1], up[2:]
        status = torch.empty(6, dtype=torch.int32, device=dev)
        (ip, inb, ie), (op, onb, oe) = _group_both(coo_src, coo_dst, num_nodes, status[:2])
        columns, read = [], 2
        for t, num in zip(given, (num_ntypes, num_etypes)):
            if t is None:
                columns.append(None)
                continue
            column = types.pop(0)
            pointer, _ = _sorted_pointer(column, num, status[read:read + 2])
            columns.append((pointer, column))
            read += 2
        status = status[:read].tolist()             # the host waits once, behind all launches
    if status.pop(0) | status.pop(0):
        raise ValueError("edge endpoint outside [0, num_nodes)")
    g = DGLGraph(ip, inb, ie, op, onb, oe, coo_src, coo_dst, None, None)
    for given_type, column, set_pointer, set_column in (
            (given[0], columns[0], g.SetNtypePointer, g.SetNtypeCOO),
            (given[1], columns[1], g.SetEtypePointer, g.SetEtypeCOO)):
        if given_type is None:
            continue
        outside, unsorted = status.pop(0), status.pop(0)
        if unsorted:
            raise ValueError("items must be sorted by type")
        if outside:
            raise ValueError("type outside [0, num_types)")
        set_pointer(column[0])
        set_column(column[1])
    return g
