"""The contraction kernels of the UVW convolution against 64-bit torch products, at tile edges."""

import pytest
import torch

pytestmark = pytest.mark.gpu
DEV = "cuda"


def make_op(in1, in2, out, dtype):
    from lunaequivariance_amd import Irreps, TensorProductConfig
    from lunaequivariance_amd.uvw_conv import LunaTPUVWConv

    a, b, c = Irreps(in1), Irreps(in2), Irreps(out)
    paths = [(i, j, k, "uvw", True) for i, (_, x) in enumerate(a) for j, (_, y) in enumerate(b)
             for k, (_, z) in enumerate(c) if z in x * y]
    return LunaTPUVWConv(TensorProductConfig(in1, in2, out, paths, shared_weights=True, internal_weights=False),
                         dtype=dtype)


def reference(op, a, w, g):
    """out, gA and gW in 64 bits."""
    rows = a.shape[0]
    out = torch.zeros(rows, op.out_dim, dtype=torch.float64, device=a.device)
    ga, gw = torch.zeros_like(a), torch.zeros_like(w)
    perm = op._perm.to(a.device)
    for blk in op.blocks:
        C, d3, m3 = blk["channels"], blk["d3"], blk["mul3"]
        lo, o = blk["a_lo"], blk["out_off"]
        A = a[:, lo:lo + C * d3].reshape(rows, C, d3)
        G = g[:, o:o + m3 * d3].reshape(rows, m3, d3)
        idx = perm[blk["w_lo"]:blk["w_lo"] + C * m3]
        W = w[idx].reshape(C, m3)
        out[:, o:o + m3 * d3] = torch.einsum("nck,cw->nwk", A, W).reshape(rows, -1)
        ga[:, lo:lo + C * d3] = torch.einsum("nwk,cw->nck", G, W).reshape(rows, -1)
        gw[idx] = torch.einsum("nck,nwk->cw", A, G).reshape(-1)
    return out, ga, gw


# Edge copies (mul2 = 2, 3), sides below, at and above a 32- or 64-wide tile, channel counts that
# are no multiple of a staged chunk, a hole in the output, and every staged degree.
LAYOUTS = [
    ("32x0e+32x1o+32x2e", "1x0e+1x1o+1x2e", "32x0e+32x1o+32x2e"),
    ("64x0e+64x1o", "1x0e+1x1o", "65x0e+64x1o"),
    ("5x0e+7x1o", "2x0e+3x1o", "33x0e+3x1o+2x2e+1x3o"),
    ("17x2e", "1x0e+1x3o", "40x5o+31x4o"),
    ("1x0e", "1x0e", "1x0e"),
]


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rows", [1, 20, 129, 2500])
@pytest.mark.parametrize("layout", LAYOUTS)
def test_the_three_products(layout, rows, dtype):
    op = make_op(*layout, dtype)
    assert op.native_contraction
    gen = torch.Generator().manual_seed(rows)
    draw = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64).to(dtype).to(DEV)  # noqa: E731
    a, w, g = draw(rows, op.aggregate_dim), draw(op.weight_numel), draw(rows, op.out_dim)
    found = [op.contraction.run(*args) for args in (("out", a, w), ("a", g, w), ("w", a, g))]
    exact = reference(op, a.double(), w.double(), g.double())
    # Rounding errors of a sum of K products are independent to first order, so its error is
    # within a few sqrt(K) eps of the sum of the products' magnitudes, in any order.
    bound = reference(op, a.double().abs(), w.double().abs(), g.double().abs())
    eps = torch.finfo(dtype).eps
    lengths = (max(b["channels"] for b in op.blocks), max(b["mul3"] for b in op.blocks), rows * 11)
    for value, want, most, length in zip(found, exact, bound, lengths):
        assert value.dtype == dtype
        assert ((value.double() - want).abs() <= 4 * length ** 0.5 * eps * most).all()


def test_derivatives_of_every_order_and_no_rows():
    op = make_op("3x0e+2x1o", "1x0e+2x1o", "2x0e+3x1o", torch.float64)
    from lunaequivariance_amd.uvw_conv import _Contract

    a = torch.randn(5, op.aggregate_dim, device=DEV, dtype=torch.float64, requires_grad=True)
    w = torch.randn(op.weight_numel, device=DEV, dtype=torch.float64, requires_grad=True)
    call = lambda *args: _Contract.apply(op.contraction, "out", *args)  # noqa: E731
    assert torch.autograd.gradcheck(call, (a, w))
    assert torch.autograd.gradgradcheck(call, (a, w))
    empty = a.detach()[:0].requires_grad_()
    out = call(empty, w)
    assert out.shape == (0, op.out_dim)
    ga, gw = torch.autograd.grad(out, (empty, w), out)
    assert ga.shape == empty.shape and not gw.count_nonzero()


def test_misuse_raises():
    op = make_op("3x0e", "1x0e", "2x0e", torch.float32)
    a = torch.randn(4, op.aggregate_dim, device=DEV)
    with pytest.raises(TypeError):
        op.contraction.run("out", a, torch.randn(op.weight_numel, device=DEV, dtype=torch.float64))
    with pytest.raises(RuntimeError):
        op.contraction.run("out", a, torch.randn(op.weight_numel))


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("rows", [3, 700])
@pytest.mark.parametrize("channels", [24, 48, 80, 96, 112, 160])
def test_widths_whose_weight_rows_cross_paths(channels, rows, dtype):
    """Tiles and chunks that hold channels of two or three paths, with and without a remainder."""
    irreps = "+".join(f"{channels}x{ir}" for ir in ("0e", "1o", "2e"))
    test_the_three_products((irreps, "1x0e+1x1o+1x2e", irreps), rows, dtype)


@pytest.mark.parametrize("dtype", [torch.float32, torch.float64])
@pytest.mark.parametrize("layout,native", [
    (("3x3o+2x0e", "1x3o+1x0e", "2x6e+4x0e+3x3o"), None),  # an output of degree 6
    (("8x0e+8x1o", "1x0e+2x1o", "5x0e+8x1o+3x1e+2x2e"), False),  # as for wide products of many rows
])
def test_library_products(monkeypatch, layout, native, dtype):
    """The contraction without the kernels, through two orders of derivatives."""
    from lunaequivariance_amd.uvw_conv import LunaTPUVWConv
    from tests.test_uvw_conv_gpu import check

    if native is None:
        assert not make_op(*layout, dtype).native_contraction
    else:
        monkeypatch.setattr(LunaTPUVWConv, "contracts_natively", lambda self, rows: native)
    check(*layout, 9, 40, dtype, True, 3, env=True, orders=2)
