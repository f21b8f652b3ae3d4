"""Derivative chains to third order on a side stream and under HIP graph capture
(the reference's ``test_combined_nondefault_stream_and_capture``,
``tests/lunatp/test_uvu_conv.py:933-995``, and the capture tests of
``tests/lunatp/test_uvw_conv.py:597-757, 913-955``).

A chain (output, its gradient with respect to every input, the gradient of
that against directions with respect to the inputs and the seed, and one
more order) runs eagerly on a non-default stream, then is captured once and
replayed three times with new inputs copied into the captured buffers, with
eager work and synchronisations between replays; every replay must equal
the eager chain on the same inputs (the same kernels in the same order:
bitwise in practice, checked to 1e-12 relative in fp64).
"""

import pytest
import torch

import lunaequivariance_amd as lunaeq
from tests.test_uvu_conv_gpu import random_graph

pytestmark = pytest.mark.gpu
DEV = "cuda"
DT = torch.float64


def all_paths(mode, in1, in2, out):
    a, b, c = lunaeq.Irreps(in1), lunaeq.Irreps(in2), lunaeq.Irreps(out)
    return [(i, j, k, mode, True) for i, (m, x) in enumerate(a) for j, (n, y) in enumerate(b)
            for k, (o, z) in enumerate(c) if z in x * y and (mode != "uuu" or m == n == o)]


def problem(mode, shared, nodes=23, edges=97, seed=0):
    ir = "4x0e+4x1o+4x2e"
    edge = ir if mode == "uuu" else "1x0e+1x1o+1x2e"
    conv = lunaeq.TensorProductConv(ir, edge, ir, all_paths(mode, ir, edge, ir), internal_weights=False,
                                    shared_weights=shared, dtype=DT)
    gen = torch.Generator().manual_seed(seed)
    src, dst = random_graph(nodes, edges, gen)
    graph = conv.create_graph(src.to(DEV), dst.to(DEV), nodes)
    return conv, graph, gen


def fresh(conv, graph, gen, shared):
    n, e = graph.num_nodes, graph.num_edges
    shapes = [(n, conv.irreps_in1.dim), (e, conv.irreps_in2.dim),
              (conv.weight_numel,) if shared else (e, conv.weight_numel), (e, 1), (n, conv.irreps_out.dim)]
    return [torch.randn(s, generator=gen, dtype=DT).to(DEV) for s in shapes]


def chain(conv, graph, x, y, w, env, g):
    """(out, first order, second order, third order) with fixed unit directions."""
    inputs = (x, y, w, env)
    out = conv(x, y, w, graph=graph, env=env)
    first = torch.autograd.grad(out, inputs, g, create_graph=True)
    second = torch.autograd.grad(first, inputs + (g,), [torch.ones_like(t) for t in first], create_graph=True,
                                 allow_unused=True)
    live = [t for t in second if t is not None and t.requires_grad]
    third = torch.autograd.grad(live, inputs, [torch.ones_like(t) for t in live], allow_unused=True)
    return [out, *first, *(t for t in second if t is not None), *(t for t in third if t is not None)]


@pytest.mark.parametrize("mode,shared", [("uvu", False), ("uuu", False), ("uvw", True), ("uvw", False)])
def test_third_order_chain_on_a_side_stream_and_in_a_graph(mode, shared):
    print(f"capture chain {mode} shared={shared}", flush=True)
    conv, graph, gen = problem(mode, shared)
    static = [t.requires_grad_() for t in fresh(conv, graph, gen, shared)]

    def run():
        return chain(conv, graph, *static)

    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            warm = run()
    torch.cuda.current_stream().wait_stream(side)
    eager = chain(conv, graph, *static)
    assert len(warm) == len(eager)
    for n, (a, b) in enumerate(zip(warm, eager)):
        torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-13, msg=f"side stream, output {n}")
    captured = torch.cuda.CUDAGraph()
    with torch.cuda.graph(captured, stream=side):
        outputs = run()
    for replay in range(3):
        new = fresh(conv, graph, gen, shared)
        with torch.no_grad():
            for dst, src in zip(static, new):
                dst.copy_(src)
        captured.replay()
        torch.cuda.synchronize()
        expected = chain(conv, graph, *(t.clone().requires_grad_() for t in new))
        assert len(outputs) == len(expected)
        for n, (a, b) in enumerate(zip(outputs, expected)):
            torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-13, msg=f"replay {replay}, output {n}")


@pytest.mark.parametrize("nodes,edges", [(23, 30), (9, 1200)])  # few edges per node; few nodes of many edges
def test_kernels_first_used_during_a_capture(nodes, edges):
    """A program that warmed up on another graph captures one whose kernels no call has loaded yet."""
    print(f"capture first use {nodes} {edges}", flush=True)
    conv, graph, gen = problem("uvu", False)
    warm = [t.requires_grad_() for t in fresh(conv, graph, gen, False)]

    def step(graph, x, y, w, env, g):
        out = conv(x, y, w, graph=graph, env=env)
        return [out, *torch.autograd.grad(out, (x, y, w, env), g)]

    src, dst = random_graph(nodes, edges, gen)
    other = conv.create_graph(src.to(DEV), dst.to(DEV), nodes)
    static = [t.requires_grad_() for t in fresh(conv, other, gen, False)]
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        for _ in range(2):
            step(graph, *warm)
    torch.cuda.current_stream().wait_stream(side)
    captured = torch.cuda.CUDAGraph()
    with torch.cuda.graph(captured):
        results = step(other, *static)
    for _ in range(3):
        with torch.no_grad():
            for t in static:
                t.copy_(torch.randn(t.shape, generator=gen, dtype=DT))
        captured.replay()
        torch.cuda.synchronize()
        for n, (a, b) in enumerate(zip(results, step(other, *static))):
            torch.testing.assert_close(a, b, rtol=1e-12, atol=1e-13, msg=f"replay, output {n}")
