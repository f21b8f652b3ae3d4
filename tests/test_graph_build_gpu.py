"""The graph sorts at the edges of their tiles, digits and scans, and the one-call C entry point,
against the torch-operation builder (whole numbers: equal)."""

import ctypes

import pytest
import torch

from lunaequivariance_amd import _native, make_graph
from tests.test_graph_gpu import DEV, assert_same_graph, random_graph, tables

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nodes,edges,hub", [
    (1, 4096, None),          # one node, one whole tile
    (255, 4097, None),        # one digit of node ids, a tile and one element
    (257, 8191, 200),         # two digits; degrees beyond one digit (hub of 4,095)
    (131071, 70000, None),    # 64 scan tiles: the most whose sums are not scanned in turn
    (131072, 140000, 65536),  # 65 scan tiles; hub of 70,000 edges (three digits)
    (5, 1, None),
])
def test_tile_digit_and_scan_edges(nodes, edges, hub):
    src, dst = random_graph(nodes, edges, nodes + edges, hub)
    assert_same_graph(src, dst, nodes)
    assert_same_graph(src, dst)


@pytest.mark.parametrize("nodes,edges,hub", [(300, 9000, 7), (140000, 70000, 3), (4, 0, None)])
def test_one_call_builder(nodes, edges, hub):
    src, dst = random_graph(nodes, edges, nodes, hub)
    ref = tables(make_graph(src, dst, nodes))
    lib, size = _native.lib(), ctypes.c_size_t()
    _native.check(lib.luna_graph_workspace(nodes, edges, ctypes.byref(size)), "workspace")
    workspace = torch.empty(size.value, dtype=torch.uint8, device=DEV)
    cap = nodes + edges // 32 + 1
    order = ("src", "dst", "dst_rowptr", "src_rowptr", "edge_ids_by_src", "edge_ids_by_dst", "node_order",
             "source_node_order", "node_tiers", "seg_rowptr", "seg_nodes", "seg_begin", "seg_end", "seg_order")
    out = {n: torch.empty(cap if n.startswith("seg_") and n != "seg_rowptr" else ref[n].numel(), dtype=torch.int32,
                          device=DEV) for n in order}
    s, d = src.to(DEV), dst.to(DEV)
    _native.check(lib.luna_graph_build(
        s.data_ptr() if edges else None, d.data_ptr() if edges else None, 64, nodes, edges,
        *(out[n].data_ptr() if out[n].numel() else None for n in order), workspace.data_ptr(), size.value,
        torch.cuda.current_stream().cuda_stream), "luna_graph_build")
    for name in order:
        expected = ref[name].to(torch.int32)
        assert torch.equal(out[name].cpu()[:expected.numel()], expected), name


def test_indices_outside_the_given_nodes_only_raise():
    """Validation reads them; the tables never index with them."""
    for src, dst in (([0, 1 << 40], [0, 1]), ([-(1 << 40), 0], [0, 1]), ([0, 0], [0, 1 << 33])):
        with pytest.raises(ValueError):
            make_graph(torch.tensor(src, device=DEV), torch.tensor(dst, device=DEV), 3)
