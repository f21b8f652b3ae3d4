"""UVW tensor-product convolution as aggregation on the HIP UVU kernels plus a contraction.

For a uvw path p (``src/lunatp/uvw_conv/``, e3nn's uvw connection) and an edge
e = (s -> t):

    msg_p[e, w, k] = sum_{u,v} Z_p[e, k, u, v] W_p[u, v, w],
    Z_p[e, k, u, v] = pw * sum_{i,j} C_ijk x[s, u, i] y[e, v, j]

and ``out[t] = sum_{e -> t} env[e] * msg[e]``.  With shared weights the sum
over edges commutes with the contraction over (u, v):

    out_p[t] = (sum_{e -> t} env[e] Z_p[e]) W_p = A_p[t] W_p

so the per-edge work is the aggregation ``A`` alone, which is a UVU
convolution whose weights are all one (a single broadcast weight row, never
read per edge) and whose output keeps every edge channel v in its own block;
it runs on the HIP UVU kernels.  The contraction with ``W_p`` then happens
once per node instead of once per edge: the paths into one output block are
contiguous columns of A, and the contraction kernels (``csrc/contract.cpp``, fp32
and fp64 matrix cores) take every block ``W_o^T [mul3, C] @ A_o [N, C, d3]``
(C = the sum of mul1 * mul2 over its paths) in one launch, reading A and
writing the output in their own layouts.  Per-edge weights cannot be
moved out of the edge sum: the same kernels aggregate over a graph whose
destinations are the edges themselves (``Z`` per edge), the per-edge
contraction is a batched GEMM, and the messages are summed at destinations.

Every piece is differentiable (the UVU autograd classes for the aggregation,
the contraction's three bilinear maps, torch for the batched GEMM and the sum),
so derivatives of every order follow.
"""

from __future__ import annotations

import ctypes
from functools import cached_property
from math import inf, prod

import torch

from . import _native
from .tracing import recording
from .cg import sparse_terms
from .graph import LunaTPGraph, make_graph
from .layout import TensorProductPaths
from .uvu_conv import LunaTPUVUConv, ConvForward, Rows


# Reductions over fewer rows than this stay one library GEMM.
SPLIT_K_MIN_ROWS = 4096


def _split_k_tn(a, b, chunks=16):
    """a^T @ b for tall a [K, M], b [K, N] as `chunks` partial GEMMs and a sum: the
    library GEMM on a long K and a small M x N output leaves most of the chip idle.
    The last K % chunks rows join with one more small GEMM (no padded copies)."""
    K = a.shape[0]
    if K < max(SPLIT_K_MIN_ROWS, chunks):
        return a.t() @ b
    step = K // chunks
    main = step * chunks
    out = torch.bmm(a[:main].reshape(chunks, step, -1).transpose(1, 2), b[:main].reshape(chunks, step, -1)).sum(0)
    if main < K:
        out = torch.addmm(out, a[main:].t(), b[main:])
    return out


class _RowsTimesWeight(torch.autograd.Function):
    """rows [K, C] @ W [C, M] whose weight gradient is a split-K GEMM.  The backward is
    written in differentiable operations, so higher derivatives compose."""

    @staticmethod
    def forward(ctx, rows, weight):
        ctx.save_for_backward(rows, weight)
        return rows @ weight

    @staticmethod
    def backward(ctx, grad):
        rows, weight = ctx.saved_tensors
        grad_rows = grad @ weight.t() if ctx.needs_input_grad[0] else None
        grad_weight = _split_k_tn(rows, grad) if ctx.needs_input_grad[1] else None
        return grad_rows, grad_weight


def _rows_times_weight(rows, weight):
    if recording():
        return rows @ weight
    return _RowsTimesWeight.apply(rows, weight)


class NativeContraction:
    """Owner of one C-ABI contraction plan (``luna_con_*``): every output block of an
    operator in one launch, on the layouts of the aggregate and of the output."""

    MAX_COMPONENTS = 11  # output blocks of degree 5; wider ones take the library products
    MAX_ROW = 1 << 23    # values of a row of A or of the output

    def __init__(self, op):
        self.adim, self.out_dim, self.weight_numel = op.aggregate_dim, op.out_dim, op.weight_numel
        self.dtype = op.compute_dtype
        bits = 64 if op.compute_dtype == torch.float64 else 32
        lines = [f"LUNACON1 {bits} {self.adim} {self.out_dim} {self.weight_numel} {len(op.blocks)}"]
        for blk in op.blocks:
            paths = [p for p in op.paths if p["out_off"] == blk["out_off"]]
            lines.append(f"{blk['out_off']} {blk['a_lo']} {blk['d3']} {blk['mul3']} {len(paths)} "
                         + " ".join(f"{p['w_off']} {p['mul1']} {p['mul2']}" for p in paths))
        covered = sum(blk["mul3"] * blk["d3"] for blk in op.blocks)
        self.out_factory = torch.empty if covered == self.out_dim else torch.zeros
        handle = ctypes.c_void_p()
        lib = _native.lib()
        _native.check(lib.luna_con_plan_create("\n".join(lines).encode(), _native.cache_dir().encode(),
                                               ctypes.byref(handle)), "luna_con_plan_create")
        self.handle = handle

    def precompile(self):
        _native.check(_native.lib().luna_con_plan_precompile(self.handle), "luna_con_plan_precompile")

    def _check(self, *tensors):
        for t in tensors:
            if not t.is_cuda or t.device != tensors[0].device:
                raise RuntimeError("UVW convolution operands must be on one GPU")
            if t.dtype != self.dtype:
                raise TypeError(f"expected {self.dtype}, got {t.dtype}")

    def run(self, kind, a, b):
        """"out": (A, W) -> out; "a": (g, W) -> gA; "w": (A, g) -> gW."""
        self._check(a, b)
        a, b = a.contiguous(), b.contiguous()
        lib, rows, stream = _native.lib(), a.shape[0], _native.stream_of(a)
        like = dict(device=a.device, dtype=a.dtype)
        if kind == "w":
            out = torch.empty((self.weight_numel,), **like)
            size = ctypes.c_size_t()
            _native.check(lib.luna_con_grad_w_workspace(self.handle, rows, ctypes.byref(size)),
                          "luna_con_grad_w_workspace")
            workspace = torch.empty((size.value,), device=a.device, dtype=torch.uint8)
            _native.check(lib.luna_con_grad_w(self.handle, a.data_ptr(), b.data_ptr(), out.data_ptr(),
                                              workspace.data_ptr(), size.value, rows, stream), "luna_con_grad_w")
            return out
        if kind == "out":
            out, call = self.out_factory((rows, self.out_dim), **like), lib.luna_con_fwd
        else:  # A's columns are covered by the blocks by construction
            out, call = torch.empty((rows, self.adim), **like), lib.luna_con_grad_a
        _native.check(call(self.handle, a.data_ptr(), b.data_ptr(), out.data_ptr(), rows, stream), "luna_con")
        return out

    def __del__(self):
        handle = getattr(self, "handle", None)
        try:
            if handle is not None and _native._lib is not None:
                _native._lib.luna_con_plan_destroy(handle)
        except Exception:  # interpreter shutdown
            pass
        self.handle = None


class _Contract(torch.autograd.Function):
    """One of the three bilinear maps of the contraction.  out, gA and gW are each linear in
    both operands, and each map's derivatives are the other two, so every order follows."""

    @staticmethod
    def forward(ctx, plan, kind, a, b):
        ctx.plan, ctx.kind = plan, kind
        ctx.save_for_backward(a, b)
        return plan.run(kind, a, b)

    @staticmethod
    def backward(ctx, r):
        a, b = ctx.saved_tensors
        plan, kind = ctx.plan, ctx.kind
        need_a, need_b = ctx.needs_input_grad[2:]
        apply = lambda *args: _Contract.apply(plan, *args)  # noqa: E731
        if kind == "out":    # (A, W), r along out
            return None, None, apply("a", r, b) if need_a else None, apply("w", a, r) if need_b else None
        if kind == "a":      # (g, W), r along A
            return None, None, apply("out", r, b) if need_a else None, apply("w", r, a) if need_b else None
        # (A, g), r along W
        return None, None, apply("a", b, r) if need_a else None, apply("out", a, r) if need_b else None


class LunaTPUVWConv:
    """Prepared UVW convolution (``src/lunatp/interface.py:370-408``)."""

    mode = "uvw_conv"
    index_mode = "uvw_conv"
    _contraction = None  # the contraction's plan, made on first use

    def __init__(self, tp, *, dtype=None, index_bits=32):
        paths = TensorProductPaths.from_tensor_product(tp)
        dtype = getattr(paths, "dtype", torch.float32) if dtype is None else dtype
        if dtype not in (torch.float32, torch.float64):
            raise ValueError(f"UVW convolution requires float32 or float64, got {dtype}")
        # Element offsets are 64-bit in every kernel, so both index widths run the
        # same kernels; graph tables are int32 (counts below 2^31).
        if index_bits not in (32, 64):
            raise ValueError(f"index_bits must be 32 or 64, got {index_bits}")
        self.tp = paths
        self.compute_dtype = dtype
        self.index_bits = index_bits
        self.weight_mode = "shared" if paths.shared_weights else "external"
        self.in1_dim, self.in2_dim, self.out_dim = paths.irreps_in1.dim, paths.irreps_in2.dim, paths.irreps_out.dim
        self.weight_numel = paths.weight_numel
        in_slices, edge_slices = paths.irreps_in1.slices(), paths.irreps_in2.slices()
        out_slices = paths.irreps_out.slices()
        self.paths = []
        specs = []
        a_off = w_off = 0
        max_channels = 1
        # Aggregate blocks in output order, so the paths into one output block are
        # contiguous columns of A and contract together.
        w_offsets, at = [], 0
        for ins in paths.instructions:
            w_offsets.append(at)
            at += prod(ins.path_shape) if ins.has_weight else 0
        order = sorted(range(len(paths.instructions)),
                       key=lambda n: out_slices[paths.instructions[n].i_out].start)
        for n in order:
            ins = paths.instructions[n]
            w_off = w_offsets[n]
            if ins.connection_mode != "uvw":
                raise ValueError(f"Only connection_mode='uvw' is supported, got {ins.connection_mode!r}.")
            if not ins.has_weight:
                raise ValueError("uvw instructions require weights")
            mul1, ir1 = paths.irreps_in1[ins.i_in1]
            mul2, ir2 = paths.irreps_in2[ins.i_in2]
            mul3, ir3 = paths.irreps_out[ins.i_out]
            if mul1 * mul2 * mul3 == 0:
                continue
            d1, d2, d3 = ir1.dim, ir2.dim, ir3.dim
            terms = sparse_terms(ir1.l, ir2.l, ir3.l, float(ins.path_weight))
            if dtype == torch.float32:
                terms = [(i, j, k, float(torch.tensor(c, dtype=torch.float32))) for i, j, k, c in terms]
            self.paths.append(dict(a_off=a_off, w_off=w_off, out_off=out_slices[ins.i_out].start, i_out=ins.i_out,
                                   mul1=mul1, mul2=mul2, mul3=mul3, d3=d3))
            for v in range(mul2):
                specs.append({
                    "x_offset": in_slices[ins.i_in1].start,
                    "y_offset": edge_slices[ins.i_in2].start + v * d2,
                    "out_offset": a_off + v * mul1 * d3,
                    "weight_offset": 0, "weight_stride": 1,
                    "channels": mul1, "d1": d1, "d2": d2, "d3": d3,
                    "l1": ir1.l, "l2": ir2.l, "l3": ir3.l, "terms": terms,
                })
            max_channels = max(max_channels, mul1)
            a_off += mul2 * mul1 * d3
        if at != self.weight_numel:
            raise ValueError(f"lowered weight_numel={at}, configuration reports {self.weight_numel}.")
        # Per output block: its columns of A as [C = sum of mul2 * mul1, d3] and the
        # weight rows in the same (path, v, u) order, gathered by one index.
        self.blocks, perm = [], []
        for p in self.paths:
            m1, m2, m3 = p["mul1"], p["mul2"], p["mul3"]
            if not self.blocks or self.blocks[-1]["out_off"] != p["out_off"]:
                self.blocks.append(dict(out_off=p["out_off"], d3=p["d3"], mul3=m3, a_lo=p["a_off"], channels=0,
                                        w_lo=len(perm)))
            block = self.blocks[-1]
            block["channels"] += m2 * m1
            for v in range(m2):
                for u in range(m1):
                    for w in range(m3):
                        perm.append(p["w_off"] + (u * m2 + v) * m3 + w)
        self._perm = torch.tensor(perm, dtype=torch.int64)
        self._perm_cache = {}
        self.aggregate_dim = a_off
        self.agg = None
        if specs:
            meta = {"in1_dim": self.in1_dim, "in2_dim": self.in2_dim, "out_dim": a_off,
                    "weight_numel": max_channels, "max_channels": max_channels, "generated_specs": specs,
                    "broadcast_weights": True}
            self.agg = LunaTPUVUConv(meta, dtype=dtype)
        self._ones = {}
        # The reference's "paths" configuration string, the constant a compiled
        # graph passes to lunatp::uvw_conv_* (built here, outside tracing).
        from .ops import paths_config

        self.torch_config = paths_config(self)

    def __getstate__(self):
        state = dict(self.__dict__)
        state["_ones"] = {}
        state["_perm_cache"] = {}
        state.pop("_contraction", None)
        return state

    @property
    def native_contraction(self) -> bool:
        """Whether the contraction kernels take rows of this width and stage every output degree."""
        return (bool(self.blocks) and max(self.aggregate_dim, self.out_dim) <= NativeContraction.MAX_ROW
                and all(blk["d3"] <= NativeContraction.MAX_COMPONENTS for blk in self.blocks))

    @property
    def contraction(self) -> NativeContraction:
        if self._contraction is None:
            self._contraction = NativeContraction(self)
        return self._contraction

    def contracts_natively(self, rows) -> bool:
        """Where the contraction kernels are at least as fast as the library products, forward
        and backward together (kernels and library, us; 20,000 rows unless given).

        fp32: lmax 2, 128 channels 997 and 1,427, 224 channels 3,168 and 3,091, 384 channels
        8,090 and 6,902 (2,000 rows: 933 and 927); lmax 3, 256 channels 10,576 and 9,852 (2,000
        rows: 1,160 and 1,293).  Scalar blocks, which the library multiplies without copies:
        256 channels 117 and 125 (60,000 rows: 331 and 237), 128 channels of 60,000 rows 105
        and 157.  fp64: lmax 1, 256 channels 1,415 and 1,564, 384 channels 3,327 and 3,018
        (2,000 rows: 389 and 522); scalars, 256 channels 246 and 199 (8,000 rows: 108 and 122).
        """
        return rows <= self._native_rows

    @cached_property
    def _native_rows(self) -> float:
        if not self.native_contraction:
            return -1
        width = max(min(blk["mul3"], blk["channels"]) for blk in self.blocks)
        gflop = 2e-9 * sum(blk["channels"] * blk["mul3"] * blk["d3"] for blk in self.blocks)  # a row
        double = self.compute_dtype == torch.float64
        if all(blk["d3"] == 1 for blk in self.blocks):
            return inf if width < 160 else (2 if double else 4) / gflop
        return inf if width < (320 if double else 224) else (15 if double else 20) / gflop

    def _unit_weights(self, like):
        key = (like.device, like.dtype)
        if key not in self._ones:
            self._ones[key] = torch.ones((1, self.agg.weight_numel), device=like.device, dtype=like.dtype)
        return self._ones[key]

    def _aggregate(self, x, y, env, graph):
        """A[t] = sum_{e -> t} env[e] Z[e] on the HIP UVU kernels (differentiable)."""
        ones = self._unit_weights(x)
        if recording():
            from . import ops

            out, _ = torch.ops.lunatp.uvu_conv_forward.default(x, y, ones, env, ops.graph_tables(graph),
                                                            graph.num_nodes, False, self.agg.torch_config)
            return out
        return ConvForward.apply(self.agg, graph, False, x, y, ones, env)

    def _contract(self, values, weight, rows):
        """out[n, o + w*d3 + k] = sum_c W[c, w] A[n, c, k] per output block; weight is the
        shared row [weight_numel] or per-row [rows, weight_numel].

        Shared weights: the contraction kernels (csrc/contract.cpp), every block in one
        launch.  Output degrees above 5 and wide products of many rows: one library 2-D
        GEMM per block over rows (n, k), [rows * d3, C] x [C, mul3].  Per-row weights: a
        batched GEMM.  The blocks are taken with one split (its backward is one
        concatenation).
        """
        if weight.dim() == 1 and self.contracts_natively(rows):
            return _Contract.apply(self.contraction, "out", values, weight)
        key = weight.device
        if key not in self._perm_cache:
            self._perm_cache[key] = self._perm.to(weight.device)
        per_row = weight.dim() == 2
        gathered = weight.index_select(-1, self._perm_cache[key])
        a_blocks = values.split([blk["channels"] * blk["d3"] for blk in self.blocks], 1)
        w_blocks = gathered.split([blk["channels"] * blk["mul3"] for blk in self.blocks], -1)
        pieces, at = [], 0
        for blk, a, W in zip(self.blocks, a_blocks, w_blocks):
            C, d3, m3 = blk["channels"], blk["d3"], blk["mul3"]
            if per_row:
                piece = torch.matmul(W.reshape(rows, C, m3).transpose(1, 2), a.reshape(rows, C, d3))
            elif d3 == 1:
                piece = _rows_times_weight(a, W.reshape(C, m3))
            else:
                rows_k = a.reshape(rows, C, d3).transpose(1, 2).reshape(rows * d3, C)
                piece = _rows_times_weight(rows_k, W.reshape(C, m3)).reshape(rows, d3, m3).transpose(1, 2)
            if blk["out_off"] > at:
                pieces.append(values.new_zeros((rows, blk["out_off"] - at)))
            pieces.append(piece.reshape(rows, m3 * d3))
            at = blk["out_off"] + m3 * d3
        if at < self.out_dim:
            pieces.append(values.new_zeros((rows, self.out_dim - at)))
        return torch.cat(pieces, 1) if len(pieces) > 1 else pieces[0]

    def _edge_graph(self, graph):
        """The graph whose destinations are the edges: node e receives edge e from src[e]."""
        rows = max(graph.num_nodes, graph.num_edges)
        key = ("uvw_edge_graph", rows)
        if key not in graph._tables:
            ids = torch.arange(graph.num_edges, device=graph.src.device, dtype=torch.int64)
            graph._tables[key] = make_graph(graph.src.to(torch.int64), ids, rows)
        return graph._tables[key]

    def run(self, x, edge_attr, weight=None, *, graph: LunaTPGraph, env=None, return_l0_feat=False):
        return lunatp_uvw_conv_func(self, x, edge_attr, weight, graph=graph, env=env,
                                    return_l0_feat=return_l0_feat)


def create_uvw_conv_operator(tp, *, dtype=None):
    return LunaTPUVWConv(tp, dtype=dtype)


def lunatp_uvw_conv_func(op, x, edge_attr, weight=None, *, graph: LunaTPGraph, env=None, return_l0_feat=False):
    """UVW messages summed at destinations (``src/lunatp/uvw_conv/interface.py:190-245``).

    x [num_nodes, in1_dim], edge_attr [num_edges, in2_dim]; weight is shared
    [weight_numel] (or [1, weight_numel]) for a shared-weight configuration
    and per-edge [num_edges, weight_numel] otherwise; env [num_edges] or
    [num_edges, 1].
    """
    if return_l0_feat:
        raise ValueError("return_l0_feat is not available for UVW convolution")
    if weight is None:
        raise ValueError("UVW convolution requires weights")
    N, E = graph.num_nodes, graph.num_edges
    if x.shape != (N, op.in1_dim) or edge_attr.shape != (E, op.in2_dim):
        raise ValueError("x / edge_attr do not match the graph and the irreps")
    x = x.contiguous()
    edge_attr = edge_attr.contiguous()
    if env is not None:
        env = env.reshape(-1).contiguous()
    if op.weight_mode == "shared":
        if weight.shape not in ((op.weight_numel,), (1, op.weight_numel)):
            raise ValueError(f"shared UVW weights must have shape ({op.weight_numel},)")
        weight = weight.reshape(-1)
    elif weight.shape != (E, op.weight_numel):
        raise ValueError(f"per-edge UVW weights must have shape ({E}, {op.weight_numel})")
    if recording():
        from .ops_paths import uvw_conv_tables

        return torch.ops.lunatp.uvw_conv_forward.default(
            x, edge_attr, weight.contiguous(), None if env is None else env.reshape(-1, 1),
            uvw_conv_tables(graph), N, op.torch_config)
    if op.agg is None:
        return x.new_zeros((N, op.out_dim))
    if op.weight_mode == "shared":
        aggregated = op._aggregate(x, edge_attr, env, graph)
        return op._contract(aggregated, weight, N)
    if isinstance(graph, Rows):
        # Every edge is its own destination (the row-wise product): no edge graph, no sum.
        return op._contract(op._aggregate(x, edge_attr, env, graph), weight.contiguous(), E)
    edges = op._edge_graph(graph)
    rows = edges.num_nodes
    xs = x if rows == N else torch.nn.functional.pad(x, (0, 0, 0, rows - N))
    per_edge = op._aggregate(xs, edge_attr, env, edges)[:E]
    messages = op._contract(per_edge, weight.contiguous(), E)
    dst = graph.dst.to(torch.int64)
    return x.new_zeros((N, op.out_dim)).index_add(0, dst, messages)


__all__ = ["LunaTPUVWConv", "create_uvw_conv_operator", "lunatp_uvw_conv_func"]
