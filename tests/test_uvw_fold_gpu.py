"""Aggregation with one weight row for every edge (UVW convolution): product sums per node in the
forward, products of seeds and weights per node in the backward, against the fp64 oracle.

lmax 3 holds 112 products in fp32 registers and falls back to the per-edge form in fp64 (lmax 2
does not); few nodes share a node's edges between waves; narrow blocks take several edges at once;
more edges than nodes and nodes without edges both occur.
"""

import pytest
import torch

from tests.test_uvw_conv_gpu import check

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("channels,lmax,nodes,edges,dtype,env", [
    (64, 3, 20, 150, torch.float32, False), (12, 3, 9, 400, torch.float32, True), (33, 2, 5, 300, torch.float32, False),
    (16, 3, 7, 90, torch.float64, True), (24, 2, 8, 500, torch.float64, False), (8, 2, 40, 25, torch.float32, True),
    (8, 4, 6, 40, torch.float32, False),
])
def test_folded_aggregation(channels, lmax, nodes, edges, dtype, env):
    irreps = [f"x{l}{'eo'[l % 2]}" for l in range(lmax + 1)]
    node, edge = ("+".join(f"{m}{ir}" for ir in irreps) for m in (channels, 1))
    check(node, edge, node, nodes, edges, dtype, True, channels, env=env, orders=2)
