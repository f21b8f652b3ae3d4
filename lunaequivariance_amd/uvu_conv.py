"""UVU tensor-product convolution: metadata lowering, operator and autograd.

Lowering follows ``build_uvu_conv_metadata``
(``src/lunatp/uvu_conv/kernels/utils.py:23-119``): every instruction and every
edge channel ``v`` becomes one path spec with offsets into x, y, out and the
per-edge weight row (``w[e, weight_offset + u * weight_stride]``, e3nn's
``[input_channel, edge_channel]`` layout), and sparse coefficient terms
``(i, j, k, cg * path_weight)``.

The operator hands the specs to the C-ABI library, which emits and compiles
gfx950 kernels for exactly this path set.  Autograd is built from two
differentiable primitives, the forward and the first-order backward
(``UVUConvForward``/``UVUConvBackward``, ``src/lunatp/uvu_conv/interface.py:210-348``).
Because the convolution is multilinear in (x, y, w, env) and linear in the
output seeds, every higher derivative is a sum of these two primitives with
some arguments replaced by their cotangents, so second and third order
derivatives run on the same kernels.
"""

from __future__ import annotations

import ctypes
from math import prod

import torch

from .tracing import recording
from . import _native
from .cg import sparse_terms
from .graph import LunaTPGraph
from .layout import TensorProductPaths
from .placement import run_with_workspace


def build_uvu_conv_metadata(tp, coefficient_dtype=torch.float32) -> dict:
    """Path specs of a UVU configuration (``uvu_conv/kernels/utils.py:23-119``)."""
    if coefficient_dtype not in (torch.float32, torch.float64):
        raise ValueError(
            f"UVU convolution coefficients require float32 or float64; got {coefficient_dtype}.")
    if tp.internal_weights:
        raise ValueError("Generated SO3 kernels require internal_weights=False.")
    if tp.shared_weights:
        raise ValueError("Generated SO3 kernels require shared_weights=False.")
    in_slices = tp.irreps_in1.slices()
    edge_slices = tp.irreps_in2.slices()
    out_slices = tp.irreps_out.slices()
    specs = []
    weight_offset = 0
    max_channels = 0
    for index, ins in enumerate(tp.instructions):
        if ins.connection_mode != "uvu":
            raise ValueError(f"Only connection_mode='uvu' is supported, got {ins.connection_mode!r}.")
        if not ins.has_weight:
            raise ValueError("Generated SO3 kernels require weighted uvu instructions.")
        mul_in, ir_in = tp.irreps_in1[ins.i_in1]
        mul_edge, ir_edge = tp.irreps_in2[ins.i_in2]
        mul_out, ir_out = tp.irreps_out[ins.i_out]
        if mul_in != mul_out:
            raise ValueError(
                f"UVU requires equal input/output multiplicities; got {mul_in} and {mul_out} "
                f"for path ({ins.i_in1}, {ins.i_in2}, {ins.i_out}).")
        if tuple(ins.path_shape) != (mul_in, mul_edge):
            raise ValueError(f"UVU expects path_shape=({mul_in}, {mul_edge}); got {ins.path_shape}.")
        max_channels = max(max_channels, mul_in)
        terms = sparse_terms(ir_in.l, ir_edge.l, ir_out.l, float(ins.path_weight))
        if coefficient_dtype == torch.float32:
            terms = [(i, j, k, float(torch.tensor(c, dtype=torch.float32))) for i, j, k, c in terms]
        for v in range(mul_edge):
            spec = {
                "x_offset": in_slices[ins.i_in1].start,
                "y_offset": edge_slices[ins.i_in2].start + v * ir_edge.dim,
                "out_offset": out_slices[ins.i_out].start,
                "weight_offset": weight_offset + v,
                "channels": mul_in,
                "d1": ir_in.dim, "d2": ir_edge.dim, "d3": ir_out.dim,
                "l1": ir_in.l, "l2": ir_edge.l, "l3": ir_out.l,
                "terms": terms,
            }
            if mul_edge != 1:
                spec["weight_stride"] = mul_edge
                spec["l0_path"] = index
            specs.append(spec)
        weight_offset += prod(ins.path_shape)
    if not specs:
        raise ValueError("No uvu instructions found.")
    if weight_offset != tp.weight_numel:
        raise ValueError(
            f"Lowered weight_numel={weight_offset}, but configuration reports {tp.weight_numel}.")
    return {
        "in1_dim": tp.irreps_in1.dim,
        "in2_dim": tp.irreps_in2.dim,
        "out_dim": tp.irreps_out.dim,
        "weight_numel": tp.weight_numel,
        "max_channels": max_channels,
        "generated_specs": specs,
    }


def l0_feature_layout(specs) -> tuple[dict, int]:
    """Column of each scalar-output path in the l0 feature matrix (``layout.py:150-170``).

    Edge copies of one instruction share a column block; paths are ordered by
    output offset.
    """
    offsets, keyed, width = {}, {}, 0
    for index, spec in sorted(enumerate(specs), key=lambda item: int(item[1]["out_offset"])):
        if int(spec["l3"]) != 0:
            continue
        key = ("instruction", int(spec["l0_path"])) if "l0_path" in spec else ("path", index)
        if key not in keyed:
            keyed[key] = width
            width += int(spec["channels"])
        offsets[index] = keyed[key]
    return offsets, width


def spec_text(meta: dict, dtype: torch.dtype) -> str:
    """Serialise path specs into the C-ABI's plan specification."""
    specs = meta["generated_specs"]
    offsets, l0_dim = l0_feature_layout(specs)
    bits = 64 if dtype == torch.float64 else 32
    head = (f"{bits} {meta['in1_dim']} {meta['in2_dim']} {meta['out_dim']} "
            f"{meta['weight_numel']} {len(specs)} {l0_dim}")
    # A broadcast weight row (one row read by every edge) needs the LUNAUVU2 header.
    parts = [f"LUNAUVU2 {head} 1" if meta.get("broadcast_weights") else f"LUNAUVU1 {head}"]
    for index, spec in enumerate(specs):
        terms = spec["terms"]
        head = (f"{spec['x_offset']} {spec['y_offset']} {spec['out_offset']} {spec['weight_offset']} "
                f"{int(spec.get('weight_stride', 1))} {spec['channels']} {spec['d1']} {spec['d2']} "
                f"{spec['d3']} {offsets.get(index, -1)} {len(terms)}")
        body = " ".join(f"{int(i)} {int(j)} {int(k)} {float(c)!r}" for i, j, k, c in terms)
        parts.append(head + (" " + body if body else ""))
    return "\n".join(parts) + "\n"


class NativePlan:
    """Owner of one C-ABI plan handle."""

    def __init__(self, text: str, edge_index_bits: int = 32):
        lib = _native.lib()
        handle = ctypes.c_void_p()
        _native.check(lib.luna_uvu_plan_create_ex(text.encode(), _native.cache_dir().encode(), edge_index_bits,
                                                  ctypes.byref(handle)), "luna_uvu_plan_create_ex")
        self.edge_index_bits = edge_index_bits
        self.handle = handle
        info = _native.PlanInfo()
        _native.check(lib.luna_uvu_plan_info(handle, ctypes.byref(info)), "luna_uvu_plan_info")
        self.info = info

    def bwd_workspace_bytes(self, nodes: int, edges: int) -> int:
        size = ctypes.c_size_t()
        _native.check(_native.lib().luna_uvu_conv_bwd_workspace(self.handle, nodes, edges, ctypes.byref(size)),
                      "luna_uvu_conv_bwd_workspace")
        return size.value

    def precompile(self, everything=False):
        """The kernels that every layer runs, or also those for small and sparse graphs and rows."""
        lib = _native.lib()
        call = lib.luna_uvu_plan_precompile_all if everything else lib.luna_uvu_plan_precompile
        _native.check(call(self.handle), "luna_uvu_plan_precompile")

    def __del__(self):
        handle = getattr(self, "handle", None)
        try:
            if handle is not None and _native._lib is not None:
                _native._lib.luna_uvu_plan_destroy(handle)
        except Exception:  # interpreter shutdown
            pass
        self.handle = None


class LunaTPUVUConv:
    """Prepared UVU convolution (``src/lunatp/interface.py:353-367``)."""

    mode = "uvu_conv"
    index_mode = "uvu_conv"

    def __init__(self, meta, *, dtype=torch.float32, index_bits=32):
        if dtype not in (torch.float32, torch.float64):
            raise ValueError("LunaTP uvu_conv requires torch.float32 or torch.float64.")
        # Element offsets are 64-bit in every kernel.  The width of the graph's
        # edge-offset tables picks the kernels (``plan_for``): int32 tables run
        # the 32-bit plan, int64 tables (graphs of 2^31 or more edges) the
        # 64-bit one, whatever ``index_bits`` says (src/lunatp/utils/layout.py:
        # 441-517 switches to wide offsets the same way).
        if index_bits not in (32, 64):
            raise ValueError(f"index_bits must be 32 or 64, got {index_bits}")
        self.meta = dict(meta)
        self.compute_dtype = dtype
        self.index_bits = index_bits
        self.in1_dim = int(meta["in1_dim"])
        self.in2_dim = int(meta["in2_dim"])
        self.out_dim = int(meta["out_dim"])
        self.weight_numel = int(meta["weight_numel"])
        self.max_channels = int(meta["max_channels"])
        self.generated_specs = list(meta["generated_specs"])
        self.l0_offsets, self.l0_dim = l0_feature_layout(self.generated_specs)
        self.spec = spec_text(self.meta, dtype)
        self._plans = {}
        from .ops import operator_config

        # JSON of the static configuration: the constant argument of the dispatcher ops.
        self.torch_config = operator_config(self)

    @property
    def plan(self) -> NativePlan:
        """The plan for int32 graph tables."""
        return self.plan_of(32)

    def plan_of(self, edge_index_bits: int) -> NativePlan:
        if edge_index_bits not in self._plans:
            self._plans[edge_index_bits] = NativePlan(self.spec, edge_index_bits)
        return self._plans[edge_index_bits]

    def plan_for(self, graph) -> NativePlan:
        """The plan whose kernels read ``graph``'s edge-offset tables."""
        return self.plan_of(edge_index_bits(graph))


    def run(self, x, edge_attr, weight, *, graph, env=None, return_l0_feat=False):
        return lunatp_uvu_conv_func(self, x, edge_attr, weight, graph=graph, env=env,
                                    return_l0_feat=return_l0_feat)

    def weight_linear(self):
        """Every uvu path is weighted: the convolution is linear in the weights."""
        return self

    def launch_forward(self, x, y, w, graph, env=None, want_l0=False):
        return run_forward(self, x, y, w, graph, env, want_l0)

    def launch_backward(self, x, y, w, graph, g, env=None, gl0=None, needs=(True, True, True, True)):
        return run_backward(self, x, y, w, graph, g, env, gl0, needs)

    def __getstate__(self):
        state = dict(self.__dict__)
        state["_plans"] = {}
        return state


def edge_index_bits(graph) -> int:
    """32 or 64: the width of the graph's edge-offset tables (dst_rowptr,
    src_rowptr, edge_ids_by_src must agree; node ids are int32)."""
    width = graph.dst_rowptr.dtype
    if graph.src_rowptr.dtype is width and graph.edge_ids_by_src.dtype is width:
        if width is torch.int32:
            return 32
        if width is torch.int64:
            return 64
    raise TypeError("graph edge-offset tables must all be int32 or all int64")


def create_uvu_conv_operator(tp_or_meta, *, dtype=None):
    """Prepared operator from a configuration or from prebuilt metadata."""
    from collections.abc import Mapping

    if not isinstance(tp_or_meta, Mapping):
        tp_or_meta = TensorProductPaths.from_tensor_product(tp_or_meta)
    if dtype is None:
        dtype = torch.float32
    elif dtype is not torch.float32 and dtype is not torch.float64:
        raise ValueError("LunaTP uvu_conv requires torch.float32 or torch.float64.")
    meta = tp_or_meta if isinstance(tp_or_meta, Mapping) else build_uvu_conv_metadata(tp_or_meta, dtype)
    if not meta["generated_specs"] or any(int(s["channels"]) <= 0 for s in meta["generated_specs"]):
        raise ValueError("UVU convolution requires positive channels for every path")
    return LunaTPUVUConv(meta, dtype=dtype)


# ---------------------------------------------------------------------------
# Kernel calls (no autograd)
# ---------------------------------------------------------------------------

_stream = _native.stream_of


def _check_tensors(op, *tensors):
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise RuntimeError("convolution kernels run on the GPU; got a CPU tensor")
        if t.dtype is not op.compute_dtype:
            raise TypeError(f"expected {op.compute_dtype}, got {t.dtype}")


def _check_device(op, graph, *tensors):
    _check_tensors(op, *tensors)
    if not graph.src.is_cuda:
        raise RuntimeError("graph tables must live on the GPU; build the graph from GPU tensors")
    if not (graph.src.dtype is graph.dst.dtype is graph.node_order.dtype is graph.source_node_order.dtype is torch.int32):
        raise TypeError("graph node-id tables (src, dst, node_order, source_node_order) must be int32")


class Rows:
    """In the place of a graph: a row-wise product, whose row b is node b, edge b and that
    edge's source.  The weight is a row per row, or one [1, weight_numel] shared by all."""

    __slots__ = ("num_nodes", "num_edges")

    def __init__(self, rows):
        self.num_nodes = self.num_edges = rows


def _rows_checked(op, x, y, w, graph, *more):
    """Checks the operands; True for a shared weight row."""
    _check_tensors(op, x, y, w, *more)
    rows = graph.num_nodes
    if x.shape != (rows, op.in1_dim):
        raise ValueError(f"x must have shape ({rows}, {op.in1_dim}); got {tuple(x.shape)}")
    shared = w.shape == (1, op.weight_numel)
    if y.shape != (rows, op.in2_dim) or not (shared or w.shape == (rows, op.weight_numel)):
        raise ValueError("edge_attr/weight rows must match the rows of x")
    return shared


def run_rows_forward(op, x, y, w, graph):
    shared = _rows_checked(op, x, y, w, graph)
    rows, plan = graph.num_nodes, op.plan
    factory = torch.zeros if plan.info.fwd_needs_zero else torch.empty
    out = factory((rows, op.out_dim), device=x.device, dtype=x.dtype)
    _native.check(_native.lib().luna_uvu_rows_fwd(plan.handle, x.data_ptr(), y.data_ptr(), w.data_ptr(), shared,
                                                  out.data_ptr(), rows, _stream(x)), "luna_uvu_rows_fwd")
    return out


def run_rows_backward(op, x, y, w, graph, g, needs):
    shared = _rows_checked(op, x, y, w, graph, g)
    rows, plan = graph.num_nodes, op.plan
    if needs[2] and op.meta.get("broadcast_weights"):
        raise ValueError("a broadcast weight row has no per-edge gradient")
    if g.shape != (rows, op.out_dim):
        raise ValueError(f"the output gradient must have shape ({rows}, {op.out_dim}); got {tuple(g.shape)}")
    gx, gy, gw = (torch.empty_like(t) if n else None for t, n in zip((x, y, w), needs))
    if not rows:
        return gx, gy, gw if gw is None else gw.zero_(), None
    size = ctypes.c_size_t()
    lib = _native.lib()
    if needs[1] or (needs[2] and shared):
        _native.check(lib.luna_uvu_rows_bwd_workspace(plan.handle, shared, rows, ctypes.byref(size)),
                      "luna_uvu_rows_bwd_workspace")
    workspace = torch.empty((size.value,), device=x.device, dtype=torch.uint8) if size.value else None
    _native.check(lib.luna_uvu_rows_bwd(plan.handle, x.data_ptr(), y.data_ptr(), w.data_ptr(), shared, g.data_ptr(),
                                        _native.ptr(gx), _native.ptr(gy), _native.ptr(gw), _native.ptr(workspace),
                                        size.value, rows, _stream(x)), "luna_uvu_rows_bwd")
    return gx, gy, gw, None


def run_forward(op, x, y, w, graph, env=None, want_l0=False):
    """out [N, out_dim] (and l0 [E, l0_dim]) from the forward kernel."""
    if isinstance(graph, Rows):
        return run_rows_forward(op, x, y, w, graph), None
    _check_device(op, graph, x, y, w, env)
    N, E = graph.num_nodes, graph.num_edges
    if x.shape != (N, op.in1_dim):
        raise ValueError(f"x must have shape ({N}, {op.in1_dim}); got {tuple(x.shape)}")
    weight_rows = 1 if op.meta.get("broadcast_weights") else E
    if y.shape != (E, op.in2_dim) or w.shape != (weight_rows, op.weight_numel):
        raise ValueError("edge_attr/weight rows must match the graph's edges")
    plan = op.plan_for(graph)
    factory = torch.zeros if plan.info.fwd_needs_zero else torch.empty
    out = factory((N, op.out_dim), device=x.device, dtype=x.dtype)
    l0 = None
    if want_l0:
        l0 = torch.empty((E, op.l0_dim), device=x.device, dtype=x.dtype)
    if N:
        _native.check(_native.lib().luna_uvu_conv_fwd(
            plan.handle, x.data_ptr(), y.data_ptr(), w.data_ptr(), _native.ptr(env),
            graph.src.data_ptr(), graph.dst_rowptr.data_ptr(), graph.node_order.data_ptr(),
            out.data_ptr(), _native.ptr(l0) if (l0 is not None and l0.numel()) else None,
            N, E, _stream(x)), "luna_uvu_conv_fwd")
    return out, l0


def run_backward(op, x, y, w, graph, g, env=None, gl0=None, needs=(True, True, True, True)):
    """(gx, gy, gw, genv) from the first-order backward kernels."""
    if isinstance(graph, Rows):
        return run_rows_backward(op, x, y, w, graph, g, needs[:3])
    _check_device(op, graph, x, y, w, env, g, gl0)
    N, E = graph.num_nodes, graph.num_edges
    plan = op.plan_for(graph)
    need_x, need_y, need_w, need_env = needs
    need_env = need_env and env is not None
    if need_w and op.meta.get("broadcast_weights"):
        raise ValueError("a broadcast weight row has no per-edge gradient")
    gx = gy = gw = genv = None
    if need_x:
        gx = torch.empty((N, op.in1_dim), device=x.device, dtype=x.dtype)
    if need_y:
        gy = torch.empty((E, op.in2_dim), device=x.device, dtype=x.dtype)
    if need_w:
        gw = torch.empty((E, op.weight_numel), device=x.device, dtype=x.dtype)
    if need_env:
        genv = torch.empty((E,), device=x.device, dtype=x.dtype)
    if N and (need_x or ((need_y or need_w or need_env) and E)):
        lib = _native.lib()
        size = plan.bwd_workspace_bytes(N, E) if (need_x or need_y or need_env) and E else 0

        def launch(workspace):
            _native.check(lib.luna_uvu_conv_bwd(
                plan.handle, x.data_ptr(), y.data_ptr(), w.data_ptr(), _native.ptr(env),
                g.data_ptr(), _native.ptr(gl0) if (gl0 is not None and gl0.numel()) else None,
                graph.src.data_ptr(), graph.dst_rowptr.data_ptr(), graph.node_order.data_ptr(),
                graph.src_rowptr.data_ptr(), graph.edge_ids_by_src.data_ptr(),
                _native.ptr(gx), _native.ptr(gy), _native.ptr(gw), _native.ptr(genv),
                workspace, size, N, E, _stream(x)), "luna_uvu_conv_bwd")

        if size:
            run_with_workspace(x.device, size, gw if gw is not None else gx, launch, place=x.dtype is torch.float32)
        else:
            launch(None)
    if gy is not None and not E:
        gy.zero_()
    return gx, gy, gw, genv


# ---------------------------------------------------------------------------
# Autograd
#
# Shared by every convolution operator: the classes call the operator's
# ``launch_forward`` / ``launch_backward`` kernels, and the higher-order rules
# only use multilinearity, which holds for the uvu and uuu connections alike.
# ---------------------------------------------------------------------------

def _contig(t):
    return None if t is None else t.contiguous()


def _add(a, b):
    if a is None:
        return b
    if b is None:
        return a
    return a + b


class ConvForward(torch.autograd.Function):
    """Differentiable forward of any convolution operator; its backward is ``ConvBackward``
    (the reference's ``UVUConvForward``, ``src/lunatp/uvu_conv/interface.py:210-286``)."""

    @staticmethod
    def forward(ctx, op, graph, want_l0, x, y, w, env):
        ctx.op, ctx.graph, ctx.want_l0 = op, graph, want_l0
        ctx.save_for_backward(x, y, w, env)
        ctx.set_materialize_grads(False)
        out, l0 = op.launch_forward(x, y, w, graph, env, want_l0)
        if want_l0:
            return out, l0
        return out

    @staticmethod
    def backward(ctx, g, gl0=None):
        x, y, w, env = ctx.saved_tensors
        op, graph = ctx.op, ctx.graph
        if g is None and gl0 is None:
            return None, None, None, None, None, None, None
        if g is None:
            g = x.new_zeros((graph.num_nodes, op.out_dim))
        needs = ctx.needs_input_grad
        gx, gy, gw, genv = conv_backward(op, graph, x, y, w, env, _contig(g), _contig(gl0),
                                         needs=(needs[3], needs[4], needs[5], needs[6]))
        return None, None, None, gx, gy, gw, genv


def conv_forward(op, graph, want_l0, x, y, w, env):
    """Differentiable forward used by the higher-order rules."""
    return ConvForward.apply(op, graph, want_l0, x, y, w, env)


class ConvBackward(torch.autograd.Function):
    """Differentiable first-order backward: (x, y, w, env, g, gl0) -> (gx, gy, gw, genv)."""

    @staticmethod
    def forward(ctx, op, graph, needs, x, y, w, env, g, gl0):
        ctx.op, ctx.graph = op, graph
        ctx.save_for_backward(x, y, w, env, g, gl0)
        ctx.set_materialize_grads(False)
        return op.launch_backward(x, y, w, graph, g, env, gl0, needs)

    @staticmethod
    def backward(ctx, rx, ry, rw, renv):
        x, y, w, env, g, gl0 = ctx.saved_tensors
        op, graph = ctx.op, ctx.graph
        need = ctx.needs_input_grad  # (op, graph, needs, x, y, w, env, g, gl0)
        want_l0 = gl0 is not None
        # Multilinear arguments and their cotangent directions.
        args = [x, y, w, env]
        dirs = [_contig(rx), _contig(ry), _contig(rw), _contig(renv) if env is not None else None]
        grads = [None, None, None, None]
        hg = hl0 = None
        for slot, direction in enumerate(dirs):
            if direction is None:
                continue
            substituted = list(args)
            substituted[slot] = direction
            # Along a weight direction only the weighted paths vary.
            sop = op.weight_linear() if slot == 2 else op
            # The scalar features do not depend on env: an env direction moves
            # only the node output, and the gl0 seed drops out of its terms.
            scalar = want_l0 and slot != 3
            if need[7] or (need[8] and scalar):
                result = conv_forward(sop, graph, scalar, *substituted)
                if scalar:
                    out, l0 = result
                    hl0 = _add(hl0, l0)
                else:
                    out = result
                hg = _add(hg, out)
            wanted = tuple(need[3 + other] and other != slot and args[other] is not None
                           for other in range(4))
            if any(wanted):
                parts = conv_backward(sop, graph, *substituted, g, gl0 if slot != 3 else None,
                                      needs=wanted)
                for other in range(4):
                    if wanted[other] and parts[other] is not None:
                        grads[other] = _add(grads[other], parts[other])
        return (None, None, None, grads[0], grads[1], grads[2], grads[3],
                hg if need[7] else None, hl0 if need[8] else None)


def conv_backward(op, graph, x, y, w, env, g, gl0, needs=(True, True, True, True)):
    needs = tuple(bool(n) for n in needs)
    if torch.is_grad_enabled():
        return ConvBackward.apply(op, graph, needs, x, y, w, env, g, gl0)
    return op.launch_backward(x, y, w, graph, g, env, gl0, needs)


def lunatp_uvu_conv_func(op, x, edge_attr, weight, *, graph: LunaTPGraph, env=None,
                         return_l0_feat=False):
    """Aggregate UVU edge messages at destination nodes (``uvu_conv/interface.py:143-204``).

    x [num_nodes, in1_dim], edge_attr [num_edges, in2_dim], weight
    [num_edges, weight_numel], env [num_edges] or [num_edges, 1].  Returns
    out [num_nodes, out_dim], or (out, l0_feat [num_edges, l0_dim]).
    """
    if weight is None:
        raise ValueError("UVU convolution requires explicit per-edge weights")
    x = x.contiguous()
    edge_attr = edge_attr.contiguous()
    weight = weight.contiguous()
    if env is not None:
        env = env.reshape(-1).contiguous()
    if recording():
        from . import ops

        out, l0 = torch.ops.lunatp.uvu_conv_forward.default(
            x, edge_attr, weight, env, ops.graph_tables(graph), graph.num_nodes, bool(return_l0_feat),
            op.torch_config)
        return (out, l0) if return_l0_feat else out
    return ConvForward.apply(op, graph, bool(return_l0_feat), x, edge_attr, weight, env)


# The reference's names for the same autograd nodes.
UVUConvForward, UVUConvBackward = ConvForward, ConvBackward

__all__ = ["ConvForward", "ConvBackward", "build_uvu_conv_metadata", "l0_feature_layout", "spec_text", "LunaTPUVUConv", "Rows",
           "create_uvu_conv_operator", "lunatp_uvu_conv_func", "run_forward", "run_backward",
           "NativePlan"]
