"""The row kernels of the uvu product (and of the row form of the uvw product) against the
fp64 oracle: row b's edge goes from and to b.

Cases sit where the kernels can go wrong: chunks of 8 to 64 channels with idle lanes, two
chunks, several rows at once with a ragged last group, more rows than workgroups, weight
rows of their own and one shared row, edge copies (strided weights), fp64 groups cut in two,
blocks that alias or leave holes.
"""

import pytest
import torch

import lunaequivariance_amd as lunaeq
from oracle.uvu_conv import conv as oracle_conv
from tests.test_rowwise_gpu import paths
from tests.test_uvu_conv_gpu import DEV, assert_close

pytestmark = pytest.mark.gpu


def full(channels, lmax, copies=1):
    """(in1, in2, out, instructions) with an output block for every path up to lmax."""
    irs = [lunaeq.Irreps(f"1x{l}{'eo'[l % 2]}")[0][1] for l in range(lmax + 1)]
    in1 = "+".join(f"{channels}x{ir}" for ir in irs)
    in2 = "+".join(f"{copies}x{ir}" for ir in irs)
    outs, ins = [], []
    for i, a in enumerate(irs):
        for j, b in enumerate(irs):
            for c in a * b:
                if c.l <= lmax:
                    ins.append((i, j, len(outs), "uvu", True))
                    outs.append(f"{channels}x{c}")
    return in1, in2, "+".join(outs), ins


def check(in1, in2, out, ins, rows, shared, dtype, needs=(True, True, True)):
    tp = lunaeq.TensorProduct(in1, in2, out, ins, shared_weights=shared, internal_weights=False, dtype=dtype)
    gen = torch.Generator().manual_seed(rows)
    draw = lambda *shape: torch.randn(*shape, generator=gen, dtype=torch.float64)  # noqa: E731
    x, y, g = draw(rows, tp.irreps_in1.dim), draw(rows, tp.irreps_in2.dim), draw(rows, tp.irreps_out.dim)
    w = draw(*((tp.weight_numel,) if shared else (rows, tp.weight_numel)))
    ids = torch.arange(rows)
    ref_in = [t.clone().requires_grad_(n) for t, n in zip((x, y, w), needs)]
    ref = oracle_conv(in1, in2, out, ins, ref_in[0], ref_in[1], ref_in[2].expand(rows, -1) if shared else ref_in[2],
                      ids, ids, rows)
    dev_in = [t.to(DEV, dtype).requires_grad_(n) for t, n in zip((x, y, w), needs)]
    act = tp(*dev_in)
    assert_close(act, ref, dtype, "forward")
    wanted = [n for n, need in enumerate(needs) if need]
    ref_grads = torch.autograd.grad(ref, [ref_in[n] for n in wanted], g)
    grads = torch.autograd.grad(act, [dev_in[n] for n in wanted], g.to(DEV, dtype))
    for n, a, r in zip(wanted, grads, ref_grads):
        assert_close(a, r, dtype, f"gradient {n}")


@pytest.mark.parametrize("channels,lmax,rows,shared,dtype", [
    (8, 1, 1, True, torch.float32), (8, 1, 6001, True, torch.float32), (16, 2, 13, False, torch.float32),
    (24, 1, 7, True, torch.float64), (32, 2, 301, True, torch.float32), (50, 2, 130, False, torch.float32),
    (64, 2, 3001, True, torch.float32), (96, 1, 33, True, torch.float32), (128, 1, 65, False, torch.float64),
    (32, 3, 41, True, torch.float64), (64, 3, 9, True, torch.float64), (130, 1, 5, True, torch.float32),
])
def test_rows_against_oracle(channels, lmax, rows, shared, dtype):
    check(*full(channels, lmax), rows, shared, dtype)


@pytest.mark.parametrize("shared", [False, True])
def test_rows_copies_aliases_and_holes(shared):
    check(*full(12, 1, copies=2), 37, shared, torch.float32)
    # Paths summed into shared outputs, an unused input block and an unused output block.
    in1, in2, out = "16x0e+16x1o+5x2e", "1x0e+1x1o", "16x0e+16x1o+3x0e"
    check(in1, in2, out, paths("uvu", "16x0e+16x1o", in2, "16x0e+16x1o"), 21, shared, torch.float32)


@pytest.mark.parametrize("needs", [(True, False, False), (False, True, False), (False, False, True), (True, False, True)])
def test_rows_subsets_of_gradients(needs):
    check(*full(16, 1), 19, True, torch.float32, needs)


@pytest.mark.parametrize("shared", [False, True])
def test_more_rows_than_waves(shared):
    """Past 2^20 waves (two chunks of channels: 2^19 rows) the first workgroups take another row."""
    rows, channels = (1 << 19) + 3, 65
    tp = lunaeq.TensorProduct(f"{channels}x0e", "1x0e", f"{channels}x0e", [(0, 0, 0, "uvu", True)], shared_weights=shared,
                              internal_weights=False)
    gen = torch.Generator(device=DEV).manual_seed(1)
    x, g = (torch.randn(rows, channels, device=DEV, generator=gen) for _ in range(2))
    y = torch.randn(rows, 1, device=DEV, generator=gen)
    w = torch.randn(*((channels,) if shared else (rows, channels)), device=DEV, generator=gen)
    ins = [t.requires_grad_() for t in (x, y, w)]
    grads = torch.autograd.grad(tp(*ins), ins, g)
    out = tp(x, y, w)
    X, Y, W, G = (t.detach().double() for t in (x, y, w, g))
    gw = G * X * Y
    for name, a, r in (("out", out, X * Y * W), ("gx", grads[0], G * Y * W), ("gy", grads[1], (G * X * W).sum(1, keepdim=True)),
                       ("gw", grads[2], gw.sum(0) if shared else gw)):
        assert_close(a, r, torch.float32, name)
