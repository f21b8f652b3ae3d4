"""Graph validation and CSR tables shared by the convolution kernels.

Restates ``make_graph`` / ``LunaTPGraph`` (``src/lunatp/graph.py:17-141``) and
``make_source_segments`` (``src/lunatp/uvu_conv/graph.py:38-99``).  Tables of
GPU inputs are built by the HIP kernels of the C-ABI library (radix sort,
scans, binary-search row pointers); tables of CPU inputs with torch
operations.  Both orderings are *stable* (equal sources keep destination
order, equal degrees keep node order), so every table is deterministic and
the two builders agree exactly.

Tables (int32; the edge-offset tables dst_rowptr, src_rowptr, edge_ids_by_src,
edge_ids_by_dst and the segment begin/end/rowptr/order are int64 when the edge
count, or nodes plus segments, reach 2^31, ``src/lunatp/graph.py:99-100``):
  src, dst           copies of the inputs (the graph owns them)
  dst_rowptr[N+1]    destination CSR over the dst-sorted edge list
  src_rowptr[N+1]    source CSR over ``edge_ids_by_src``
  edge_ids_by_src[E] edge ids ordered by source
  edge_ids_by_dst[E] identity (edges are dst-sorted)
  node_order[N]      nodes by descending in-degree (launch order, forward)
  source_node_order  nodes by descending out-degree (launch order, backward)
  node_tiers[3]      prefix lengths of node_order covering 1/4, 2/4, 3/4 of edges
  source_segments    source-CSR chunks of at most 32 edges
"""

from __future__ import annotations

from dataclasses import dataclass, field
from operator import index

import torch

SOURCE_SEGMENT_EDGES = 32
# Edge offsets at or above this take int64 tables (the reference's rule,
# src/lunatp/graph.py:99-100: edges or nodes + edges / 32 segments >= 2^31).
WIDE_OFFSETS = 1 << 31


def wide_offsets(num_nodes: int, num_edges: int) -> bool:
    """True when a graph's edge-offset tables must be int64."""
    return max(num_edges, num_nodes + num_edges // SOURCE_SEGMENT_EDGES) >= WIDE_OFFSETS


@dataclass(frozen=True)
class SourceSegmentTables:
    """Source-CSR segments of at most ``SOURCE_SEGMENT_EDGES`` edges.

    ``nodes`` owns each segment, ``begin``/``end`` index ``edge_ids_by_src``,
    ``rowptr`` maps a node to its segments and ``order`` is a launch permutation
    (longest segments of the highest-degree nodes first).
    """

    nodes: torch.Tensor
    begin: torch.Tensor
    end: torch.Tensor
    rowptr: torch.Tensor
    order: torch.Tensor


@dataclass(frozen=True)
class LunaTPGraph:
    """Prepared topology; tables are never modified after construction."""

    src: torch.Tensor
    dst: torch.Tensor
    num_nodes: int
    dst_rowptr: torch.Tensor
    src_rowptr: torch.Tensor
    edge_ids_by_src: torch.Tensor
    edge_ids_by_dst: torch.Tensor
    node_order: torch.Tensor | None = None
    source_node_order: torch.Tensor | None = None
    node_tiers: torch.Tensor | None = None
    source_segments: SourceSegmentTables | None = None
    _tables: dict = field(default_factory=dict, init=False, repr=False, compare=False)

    @property
    def num_edges(self) -> int:
        return int(self.src.numel())

    def to(self, device) -> "LunaTPGraph":
        """Copy every table to ``device``."""
        def move(t):
            return None if t is None else t.to(device)
        seg = self.source_segments
        return LunaTPGraph(
            src=move(self.src), dst=move(self.dst), num_nodes=self.num_nodes,
            dst_rowptr=move(self.dst_rowptr), src_rowptr=move(self.src_rowptr),
            edge_ids_by_src=move(self.edge_ids_by_src), edge_ids_by_dst=move(self.edge_ids_by_dst),
            node_order=move(self.node_order), source_node_order=move(self.source_node_order),
            node_tiers=move(self.node_tiers),
            source_segments=None if seg is None else SourceSegmentTables(
                *(move(t) for t in (seg.nodes, seg.begin, seg.end, seg.rowptr, seg.order))),
        )


def make_source_segments(src_rowptr: torch.Tensor, wide: bool = False) -> SourceSegmentTables:
    """Split every source row into chunks of at most 32 edges (``uvu_conv/graph.py:38-99``).

    Isolated nodes keep one empty segment so the segment CSR covers every node.
    ``wide`` keeps begin/end/rowptr/order in int64 (nodes stay int32).
    """
    rowptr = src_rowptr.to(torch.int64)
    degree = rowptr[1:] - rowptr[:-1]
    count = ((degree + SOURCE_SEGMENT_EDGES - 1) // SOURCE_SEGMENT_EDGES).clamp_min(1)
    seg_rowptr = torch.zeros(degree.numel() + 1, dtype=torch.int64, device=rowptr.device)
    torch.cumsum(count, 0, out=seg_rowptr[1:])
    total = int(seg_rowptr[-1].item())
    nodes = torch.repeat_interleave(torch.arange(degree.numel(), device=rowptr.device), count,
                                    output_size=total)
    local = torch.arange(total, device=rowptr.device) - torch.repeat_interleave(
        seg_rowptr[:-1], count, output_size=total)
    begin = rowptr[nodes] + SOURCE_SEGMENT_EDGES * local
    end = torch.minimum(begin + SOURCE_SEGMENT_EDGES, rowptr[nodes + 1])
    by_degree = torch.argsort(degree[nodes], descending=True, stable=True)
    order = by_degree[torch.argsort((end - begin)[by_degree], descending=True, stable=True)]
    i32 = torch.int32
    off = torch.int64 if wide else i32
    return SourceSegmentTables(nodes.to(i32), begin.to(off), end.to(off), seg_rowptr.to(off), order.to(off))


def make_graph(src: torch.Tensor, dst: torch.Tensor, num_nodes: int | None = None) -> LunaTPGraph:
    """Build the topology shared by all convolution layers.

    ``src``/``dst`` are ``[edges]`` or ``[edges, 1]`` int32/int64 with ``dst``
    sorted ascending; edge data must follow the same order.  Errors follow
    ``src/lunatp/graph.py:64-98``.
    """
    if src.ndim == 2 and src.shape[1] == 1:
        src = src.squeeze(-1)
    if dst.ndim == 2 and dst.shape[1] == 1:
        dst = dst.squeeze(-1)
    if src.ndim != 1 or dst.ndim != 1 or src.shape != dst.shape:
        raise ValueError("src and dst must have equal shape [edges] or [edges, 1].")
    if src.dtype not in (torch.int32, torch.int64) or dst.dtype not in (torch.int32, torch.int64):
        raise TypeError("graph indices must be int32 or int64.")
    if num_nodes is not None and not isinstance(num_nodes, int):
        num_nodes = index(num_nodes)
    num_edges = src.numel()
    if src.is_cuda:
        return _make_graph_device(src, dst, num_nodes)
    return _make_graph_torch(src, dst, num_nodes)


def _make_graph_torch(src: torch.Tensor, dst: torch.Tensor, num_nodes) -> LunaTPGraph:
    """Tables from torch operations on the inputs' device: the builder of CPU
    graphs, and of device graphs whose edge offsets need int64."""
    num_edges = src.numel()
    required = 0
    if num_edges:
        src_min, src_max = torch.aminmax(src)
        dst_min, dst_max = torch.aminmax(dst)
        low = min(int(src_min), int(dst_min))
        required = max(int(src_max), int(dst_max)) + 1
        if low < 0:
            raise ValueError("graph indices must be nonnegative.")
        if num_edges > 1 and bool((dst[1:] < dst[:-1]).any()):
            raise ValueError(
                "dst must be sorted in ascending order; src and edge data must follow the same order.")
    num_nodes = _check_nodes(num_nodes, required, num_edges)

    device = src.device
    i32 = torch.int32
    wide = wide_offsets(num_nodes, num_edges)
    off = torch.int64 if wide else i32
    src64, dst64 = src.to(torch.int64), dst.to(torch.int64)
    src_deg = torch.bincount(src64, minlength=num_nodes)
    dst_deg = torch.bincount(dst64, minlength=num_nodes)
    src_rowptr = torch.zeros(num_nodes + 1, dtype=off, device=device)
    dst_rowptr = torch.zeros(num_nodes + 1, dtype=off, device=device)
    if num_nodes:
        torch.cumsum(src_deg, 0, dtype=off, out=src_rowptr[1:])
        torch.cumsum(dst_deg, 0, dtype=off, out=dst_rowptr[1:])
    node_order = torch.argsort(dst_deg, descending=True, stable=True).to(i32)
    source_node_order = torch.argsort(src_deg, descending=True, stable=True).to(i32)
    if num_nodes and num_edges:
        cumulative = dst_deg[node_order.long()].cumsum(0)
        thresholds = torch.arange(1, 4, device=device, dtype=torch.int64) * num_edges // 4
        node_tiers = (torch.searchsorted(cumulative, thresholds) + 1).to(i32)
    else:
        node_tiers = torch.full((3,), num_nodes, device=device, dtype=i32)
    graph = LunaTPGraph(
        src=src.to(dtype=i32, copy=True, memory_format=torch.contiguous_format),
        dst=dst.to(dtype=i32, copy=True, memory_format=torch.contiguous_format),
        num_nodes=num_nodes,
        dst_rowptr=dst_rowptr,
        src_rowptr=src_rowptr,
        edge_ids_by_src=_stable_order(src64, src_rowptr, num_nodes).to(off),
        edge_ids_by_dst=torch.arange(num_edges, device=device, dtype=off),
        node_order=node_order,
        source_node_order=source_node_order,
        node_tiers=node_tiers,
        source_segments=make_source_segments(src_rowptr, wide),
    )
    return graph


SORT_CHUNK = 1 << 30  # largest count one torch sort takes here (its limit is 2^31 - 1)


def _stable_order(keys: torch.Tensor, rowptr: torch.Tensor, num_nodes: int) -> torch.Tensor:
    """Edge ids ordered by key, equal keys in edge order (a stable argsort).

    One torch sort when the edges fit it; otherwise a stable counting sort over
    chunks of ``SORT_CHUNK`` edges: each chunk is sorted on its own, and an
    edge lands at rowptr[key] + (edges of that key in earlier chunks) + (its
    rank among the chunk's edges of that key)."""
    num_edges = keys.numel()
    if num_edges <= SORT_CHUNK:
        return torch.argsort(keys, stable=True)
    device = keys.device
    order = torch.empty(num_edges, dtype=torch.int64, device=device)
    before = torch.zeros(num_nodes, dtype=torch.int64, device=device)  # edges of each key in earlier chunks
    base = rowptr[:-1].to(torch.int64)
    for start in range(0, num_edges, SORT_CHUNK):
        chunk = keys[start:start + SORT_CHUNK]
        local = torch.argsort(chunk, stable=True)
        sorted_keys = chunk[local]
        counts = torch.bincount(chunk, minlength=num_nodes)
        first = torch.cumsum(counts, 0) - counts  # first sorted position of each key in the chunk
        rank = torch.arange(chunk.numel(), device=device) - first[sorted_keys]
        order[base[sorted_keys] + before[sorted_keys] + rank] = local + start
        before += counts
    return order


def _check_nodes(num_nodes, required, num_edges):
    if num_nodes is None:
        num_nodes = required
    if num_nodes < required:
        raise ValueError(
            f"num_nodes={num_nodes} must be nonnegative and at least {required} for the supplied indices.")
    if num_nodes >= (1 << 31):
        raise OverflowError("graph node count exceeds signed int32 capacity.")
    return num_nodes


def _make_graph_device(src: torch.Tensor, dst: torch.Tensor, num_nodes) -> LunaTPGraph:
    """Tables of a device graph from the HIP kernels of the C-ABI library
    (``luna_graph_scan`` / ``luna_graph_finish``; the reference's topology
    extension, ``src/lunatp/utils/graph.py:142-846``).  The indices are always
    validated (one read-back of min, max and sortedness, together with the
    segment count and the largest degrees), also when ``num_nodes`` is given,
    because every later kernel indexes with them."""
    import ctypes

    from . import _native

    if src.dtype != dst.dtype:
        dst = dst.to(src.dtype)
    src, dst = src.contiguous(), dst.contiguous()
    bits = 64 if src.dtype == torch.int64 else 32
    E = num_edges = src.numel()
    if wide_offsets(num_nodes or 0, num_edges):
        return _make_graph_torch(src, dst, num_nodes)
    device = src.device
    lib = _native.lib()
    _native.check(lib.luna_graph_precompile(_native.cache_dir().encode()), "luna_graph_precompile")
    stream = torch.cuda.current_stream(device).cuda_stream
    status = torch.empty(8, dtype=torch.int64, device=device)

    def validated(low, high, unsorted):
        """The nodes the indices require."""
        if low < 0:
            raise ValueError("graph indices must be nonnegative.")
        if unsorted:
            raise ValueError(
                "dst must be sorted in ascending order; src and edge data must follow the same order.")
        return high + 1

    if num_nodes is None:
        required = 0
        if num_edges:
            _native.check(lib.luna_graph_bounds(src.data_ptr(), dst.data_ptr(), bits, num_edges, status.data_ptr(),
                                                stream), "luna_graph_bounds")
            required = validated(*status[:3].tolist())
        num_nodes = _check_nodes(None, required, num_edges)
        if wide_offsets(num_nodes, num_edges):
            # int64 edge offsets: torch's sorts and scans on the device (the HIP
            # builder's radix sort carries int32 edge ids).
            return _make_graph_torch(src, dst, num_nodes)
    elif num_nodes < 0:
        return _check_nodes(num_nodes, 0, num_edges)
    N = num_nodes
    new = lambda n: torch.empty(n, dtype=torch.int32, device=device)  # noqa: E731
    t = {name: new(n) for name, n in (
        ("src", E), ("dst", E), ("dst_rowptr", N + 1), ("src_rowptr", N + 1), ("edge_ids_by_src", E),
        ("edge_ids_by_dst", E), ("node_order", N), ("source_node_order", N), ("node_tiers", 3),
        ("seg_rowptr", N + 1))}
    size = ctypes.c_size_t()
    _native.check(lib.luna_graph_workspace(N, E, ctypes.byref(size)), "luna_graph_workspace")
    workspace = torch.empty(max(size.value, 1), dtype=torch.uint8, device=device)
    scratch = (workspace.data_ptr(), size.value, stream)
    address = lambda *names: (t[name].data_ptr() if t[name].numel() else None for name in names)  # noqa: E731
    _native.check(lib.luna_graph_scan(
        src.data_ptr() if E else None, dst.data_ptr() if E else None, bits, N, E,
        *address("src", "dst", "dst_rowptr", "src_rowptr", "edge_ids_by_src", "edge_ids_by_dst", "seg_rowptr"),
        status.data_ptr(), *scratch), "luna_graph_scan")
    low, high, unsorted, segments, most_in, most_out, _, _ = status.tolist()
    _check_nodes(N, validated(low, high, unsorted) if E else 0, num_edges)
    t.update({name: new(segments) for name in ("seg_nodes", "seg_begin", "seg_end", "seg_order")})
    _native.check(lib.luna_graph_finish(
        *address("dst_rowptr", "src_rowptr", "seg_rowptr"), N, E, max(most_in, most_out), segments,
        *address("node_order", "source_node_order", "node_tiers", "seg_nodes", "seg_begin", "seg_end", "seg_order"),
        *scratch), "luna_graph_finish")
    return LunaTPGraph(
        src=t["src"], dst=t["dst"], num_nodes=N,
        dst_rowptr=t["dst_rowptr"], src_rowptr=t["src_rowptr"],
        edge_ids_by_src=t["edge_ids_by_src"], edge_ids_by_dst=t["edge_ids_by_dst"],
        node_order=t["node_order"], source_node_order=t["source_node_order"], node_tiers=t["node_tiers"],
        source_segments=SourceSegmentTables(
            t["seg_nodes"], t["seg_begin"], t["seg_end"], t["seg_rowptr"], t["seg_order"]),
    )


__all__ = ["LunaTPGraph", "SourceSegmentTables", "make_graph", "make_source_segments", "wide_offsets",
           "SOURCE_SEGMENT_EDGES", "WIDE_OFFSETS"]
