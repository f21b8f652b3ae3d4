"""UVU kernels that take several edges per wave (narrow channel blocks) or several waves per node
(few nodes, many edges each) against the fp64 oracle.

Channel counts stand at the edges of the chunk widths (8, 16, 32, 64) and of two and three chunks;
graphs have a node without edges and row lengths that are no multiple of the edges taken at once.
"""

import pytest
import torch

from tests.conftest import mace_irreps
from tests.test_uvu_conv_gpu import all_uvu_instructions, check_orders, inputs, make_conv, random_graph

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("channels", [1, 8, 9, 17, 32, 33, 64, 66, 96, 130])
@pytest.mark.parametrize("nodes,edges", [(30, 200), (9, 1000)])
def test_first_order_over_chunk_widths(channels, nodes, edges, dtype):
    gen = torch.Generator().manual_seed(channels + edges)
    in1, sh, out, instructions = mace_irreps(channels, 2 if channels > 40 else 3)
    conv = make_conv(in1, sh, out, instructions, dtype)
    src, dst = random_graph(nodes - 1, edges, gen)
    x, y, w = inputs(conv, nodes, edges, dtype, gen)
    check_orders(conv, in1, sh, out, instructions, x, y, w, src, dst, nodes, dtype, gen, orders=1)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("channels,nodes,edges", [(12, 20, 150), (24, 5, 700), (64, 6, 900), (5, 6, 1100)])
def test_options_and_higher_orders(channels, nodes, edges, dtype):
    """env, scalar features, edge copies and summed output blocks (several launches)."""
    gen = torch.Generator().manual_seed(channels)
    in1, sh = f"{channels}x0e+{channels}x1o", "2x0e+1x1o"
    out = f"{channels}x0e+{channels}x1o"
    instructions = all_uvu_instructions(in1, sh, out)
    conv = make_conv(in1, sh, out, instructions, dtype)
    src, dst = random_graph(nodes, edges, gen)
    x, y, w = inputs(conv, nodes, edges, dtype, gen)
    env = torch.rand(edges, generator=gen, dtype=torch.float64)
    check_orders(conv, in1, sh, out, instructions, x, y, w, src, dst, nodes, dtype, gen, env=env, l0=True, orders=2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("channels,degree", [(8, 2), (12, 2), (32, 3)])
@pytest.mark.parametrize("more", [0, 1])
def test_both_sides_of_few_edges_per_node(channels, degree, more, dtype):
    """The most edges that are taken one at a time, and one more."""
    nodes, gen = 30, torch.Generator().manual_seed(channels + more)
    edges = degree * nodes + more
    in1, sh, out, instructions = mace_irreps(channels, 2)
    conv = make_conv(in1, sh, out, instructions, dtype)
    src, dst = random_graph(nodes - 1, edges, gen)
    x, y, w = inputs(conv, nodes, edges, dtype, gen)
    env = torch.rand(edges, generator=gen, dtype=torch.float64)
    check_orders(conv, in1, sh, out, instructions, x, y, w, src, dst, nodes, dtype, gen, env=env, l0=True, orders=2)
