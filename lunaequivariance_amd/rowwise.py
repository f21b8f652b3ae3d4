"""Row-wise UVU and UUU tensor products on the convolution kernels.

A row-wise product (``TensorProduct``, ``src/modules/tensorproduct.py:19-116``;
the reference's ``LunaTPUVU`` / ``LunaTPUUU``, ``src/lunatp/interface.py:265-307``)
is the convolution over the identity graph: row b is node b, edge b and the
destination of edge b.  UVU runs row kernels of the same plan, which read a
shared weight row once and sum its gradient; UUU runs the convolution kernels
with every segment holding one edge and shared weights ``[weight_numel]``
broadcast to every row.  UVU takes matrices ``[B, dim]``; UUU also broadcasts
leading batch dimensions of x, y and per-row weights, as the reference does.
"""

from __future__ import annotations

from copy import copy

import torch

from .tracing import recording
from .graph import make_graph
from .layout import TensorProductPaths


class LunaTPRows:
    """Prepared row-wise uvu or uuu product."""

    def __init__(self, tp, *, dtype=torch.float32):
        paths = TensorProductPaths.from_tensor_product(tp)
        modes = {ins.connection_mode for ins in paths.instructions}
        if len(modes) != 1 or not modes <= {"uvu", "uuu"}:
            raise ValueError("row-wise products here take one connection mode: uvu or uuu")
        self.mode = modes.pop()
        if dtype not in (torch.float32, torch.float64):
            raise ValueError(f"{self.mode} requires float32 or float64, got {dtype}")
        self.compute_dtype = dtype
        self.tp = paths
        self.index_mode = self.mode
        self.index_bits = 32
        self.shared_weights = bool(paths.shared_weights)
        self.weight_mode = "shared" if self.shared_weights else "external"
        # The convolution lowering takes per-edge weights; shared rows are broadcast at run time.
        flat = copy(paths)
        flat.shared_weights = False
        flat.internal_weights = False
        if self.mode == "uvu":
            from .uvu_conv import create_uvu_conv_operator

            self.conv = create_uvu_conv_operator(flat, dtype=dtype)
        else:
            from .uuu_conv import create_uuu_conv_operator

            self.conv = create_uuu_conv_operator(flat, dtype=dtype)
        self.weight_numel = self.conv.weight_numel
        self.out_dim = self.conv.out_dim
        self._identity = {}
        # The reference's "paths" configuration string, the constant a compiled
        # graph passes to lunatp::uvu_* / lunatp::uuu_* (built here, outside tracing).
        from .ops import paths_config

        self.torch_config = paths_config(self)

    def identity_graph(self, rows, device):
        key = (rows, str(device))
        if key not in self._identity:
            ids = torch.arange(rows, device=device)
            self._identity = {key: make_graph(ids, ids, rows)}
        return self._identity[key]

    def run(self, x, y, weight=None):
        if self.mode == "uuu" and (x.ndim != 2 or y.ndim != 2 or x.shape[0] != y.shape[0]
                                   or (weight is not None and weight.ndim > 1
                                       and weight.shape[:-1] != x.shape[:-1])):
            return self._run_broadcast(x, y, weight)
        if x.ndim != 2 or y.ndim != 2 or x.shape[0] != y.shape[0]:
            raise ValueError(f"{self.mode} row-wise inputs must be matrices with the same rows")
        if recording():
            if weight is None:
                raise TypeError(f"{self.mode} under torch.compile takes an explicit weight tensor")
            forward = getattr(torch.ops.lunatp, f"{self.mode}_forward").default
            return forward(x.contiguous(), y.contiguous(), weight.contiguous(), self.torch_config)
        rows = x.shape[0]
        shared = weight is not None and weight.shape in ((self.weight_numel,), (1, self.weight_numel))
        if self.mode == "uvu":
            from .uvu_conv import Rows

            return self.conv.run(x, y, weight.reshape(1, -1) if shared else weight, graph=Rows(rows))
        if shared:
            weight = weight.reshape(1, -1).expand(rows, -1)
        graph = self.identity_graph(rows, x.device)
        return self.conv.run(x, y, weight, graph=graph)

    def _run_broadcast(self, x, y, weight):
        """UUU with leading batch dimensions broadcast as in PyTorch
        (``docs/operators/tensor_product.md:48-54``): flatten, run, reshape."""
        shared = weight is None or weight.ndim == 1
        shapes = [x.shape[:-1], y.shape[:-1]] + ([] if shared else [weight.shape[:-1]])
        lead = torch.broadcast_shapes(*shapes)
        flat = lambda t: t.expand(*lead, t.shape[-1]).reshape(-1, t.shape[-1])  # noqa: E731
        out = self.run(flat(x), flat(y), weight if shared else flat(weight))
        return out.reshape(*lead, out.shape[-1])

    def __getstate__(self):
        state = dict(self.__dict__)
        state["_identity"] = {}
        return state


__all__ = ["LunaTPRows"]
