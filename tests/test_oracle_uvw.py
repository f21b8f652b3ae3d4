"""CPU oracle of the shared-weight UVW tensor product (no GPU)."""

import math

import numpy as np
import pytest
import torch

from oracle.uvu_conv import parse_irreps
from oracle.uvw import uvw_path_weights, uvw_tensor_product
from oracle.wigner import wigner_3j
from tests.test_oracle_conv import block_diag_d, rotation


def uvw_instructions(in1, in2, out):
    a, b, c = parse_irreps(in1), parse_irreps(in2), parse_irreps(out)
    return [(i, j, k, "uvw", True) for i, (_, l1, p1) in enumerate(a) for j, (_, l2, p2) in enumerate(b)
            for k, (_, l3, p3) in enumerate(c) if abs(l1 - l2) <= l3 <= l1 + l2 and p1 * p2 == p3]


def brute(in1, in2, out, instructions, x, y, w):
    a, b, c = parse_irreps(in1), parse_irreps(in2), parse_irreps(out)
    off = lambda irreps: np.cumsum([0] + [m * (2 * l + 1) for m, l, _ in irreps])
    xo, yo, oo = off(a), off(b), off(c)
    weights = uvw_path_weights(a, b, c, instructions)
    result = np.zeros((x.shape[0], oo[-1]))
    w_off = 0
    for (i1, i2, io, *_), pw in zip(instructions, weights):
        (m1, l1, _), (m2, l2, _), (m3, l3, _) = a[i1], b[i2], c[io]
        cg = wigner_3j(l1, l2, l3)
        for bb in range(x.shape[0]):
            for u in range(m1):
                for v in range(m2):
                    for ww in range(m3):
                        wt = w[w_off + (u * m2 + v) * m3 + ww]
                        for i in range(2 * l1 + 1):
                            for j in range(2 * l2 + 1):
                                for k in range(2 * l3 + 1):
                                    if cg[i, j, k] == 0:
                                        continue
                                    result[bb, oo[io] + ww * (2 * l3 + 1) + k] += (
                                        pw * cg[i, j, k] * wt * x[bb, xo[i1] + u * (2 * l1 + 1) + i]
                                        * y[bb, yo[i2] + v * (2 * l2 + 1) + j])
        w_off += m1 * m2 * m3
    return result


def test_uvw_oracle_matches_brute_force():
    in1, in2, out = "2x0e+2x1o", "1x0e+2x1o", "3x0e+2x1o+1x1e"
    instructions = uvw_instructions(in1, in2, out)
    gen = torch.Generator().manual_seed(0)
    x = torch.randn(3, 8, generator=gen, dtype=torch.float64)
    y = torch.randn(3, 7, generator=gen, dtype=torch.float64)
    wn = sum(parse_irreps(in1)[i][0] * parse_irreps(in2)[j][0] * parse_irreps(out)[k][0]
             for i, j, k, *_ in instructions)
    w = torch.randn(wn, generator=gen, dtype=torch.float64)
    dense = uvw_tensor_product(in1, in2, out, instructions, x, y, w)
    assert np.allclose(dense.numpy(), brute(in1, in2, out, instructions, x.numpy(), y.numpy(), w.numpy()),
                       atol=1e-12)


def test_uvw_path_weights_match_package():
    from lunaequivariance_amd import TensorProductConfig

    in1 = out = "4x0e+4x1o+4x2e"
    in2 = "1x0e+1x1o+1x2e"
    instructions = uvw_instructions(in1, in2, out)
    tp = TensorProductConfig(in1, in2, out, instructions, shared_weights=True)
    expected = uvw_path_weights(parse_irreps(in1), parse_irreps(in2), parse_irreps(out), instructions)
    assert [i.path_weight for i in tp.instructions] == pytest.approx(expected, rel=1e-14)
    assert tp.weight.shape == (11 * 16,)


def test_uvw_oracle_equivariance():
    in1 = out = "3x0e+3x1o+3x2e"
    in2 = "1x0e+1x1o+1x2e"
    instructions = uvw_instructions(in1, in2, out)
    gen = torch.Generator().manual_seed(2)
    x = torch.randn(4, 27, generator=gen, dtype=torch.float64)
    y = torch.randn(4, 9, generator=gen, dtype=torch.float64)
    w = torch.randn(len(instructions) * 9, generator=gen, dtype=torch.float64)
    R = rotation(5)
    rng = np.random.default_rng(6)
    D1, D2 = block_diag_d(in1, R, rng), block_diag_d(in2, R, rng)
    out_plain = uvw_tensor_product(in1, in2, out, instructions, x, y, w)
    out_rot = uvw_tensor_product(in1, in2, out, instructions, x @ D1.T, y @ D2.T, w)
    assert torch.allclose(out_rot, out_plain @ D1.T, atol=1e-10)


def test_uvw_plan_compiles_without_gpu(tmp_path, monkeypatch):
    """The matrix-core kernels of the config-5 layer are emitted and compiled for gfx950."""
    import lunaequivariance_amd as lunaeq

    monkeypatch.setenv("LUNAEQ_AMD_CACHE", str(tmp_path))
    ir, sh = "64x0e+64x1o+64x2e", "1x0e+1x1o+1x2e"
    tp = lunaeq.TensorProduct(ir, sh, ir, uvw_instructions(ir, sh, ir), shared_weights=True,
                              internal_weights=True)
    assert tp.weight_numel == 45056
    tp.op.plan.precompile()
    assert len(list(tmp_path.glob("uvw_*.co"))) == 3
    # fp64 and per-row weights take the row form of the UVW convolution
    double = lunaeq.TensorProduct(ir, sh, ir, uvw_instructions(ir, sh, ir), shared_weights=True,
                                  internal_weights=True, dtype=torch.float64)
    assert double.op.rows_op is not None and double.op.rows_op.agg.spec.startswith("LUNAUVU2 64")
    per_row = lunaeq.TensorProduct(ir, sh, ir, uvw_instructions(ir, sh, ir), shared_weights=False,
                                   internal_weights=False)
    assert per_row.op.rows_op is not None and per_row.op.weight_mode == "external"


@pytest.mark.parametrize("in1,in2,out,weights", [
    ("64x0e", "1x1o", "64x1o", [0.0]),                                   # one path, l1 < l3
    ("64x0e", "1x1o", "64x1o", [1.0]),
    ("16x0e+16x1o", "1x0e+1x1o", "16x0e+16x1o+16x2e", [1.0, 0.0, 0.0, 1.0, 0.0]),  # beside weighted paths
    ("10x0e+6x1o", "2x1o", "9x0e+7x1o+5x2e", [0.0, 0.0, 0.0]),           # unaligned rows, mul2 = 2
])
def test_uvw_plan_compiles_with_paths_of_weight_zero(tmp_path, monkeypatch, in1, in2, out, weights):
    import lunaequivariance_amd as lunaeq

    monkeypatch.setenv("LUNAEQ_AMD_CACHE", str(tmp_path))
    paths = uvw_instructions(in1, in2, out)
    assert len(paths) == len(weights)
    tp = lunaeq.TensorProduct(in1, in2, out, [(*p, w) for p, w in zip(paths, weights)], shared_weights=True,
                              internal_weights=False)
    tp.op.plan.precompile()
    assert len(list(tmp_path.glob("uvw_*.co"))) == 3


# Hand-computed uvw normalisation, the formula of the reference's
# src/lunatp/utils/layout.py:339-367 with fan = mul1 * mul2 for uvw paths.
# Config 5 ("64x0e+64x1o+64x2e" x "1x0e+1x1o+1x2e" -> same, fully connected,
# component irreps, element paths): fan 64 * 1 per path;
#   0e <- (0e,0e), (1o,1o), (2e,2e):            alpha = 1 / (3 * 64)
#   1o <- (0e,1o), (1o,0e), (1o,2e), (2e,1o):   alpha = 3 / (4 * 64)
#   2e <- (0e,2e), (1o,1o), (2e,0e), (2e,2e):   alpha = 5 / (4 * 64)
CFG5_EXPECTED = {0: math.sqrt(1 / 192), 1: math.sqrt(3 / 256), 2: math.sqrt(5 / 256)}


def _cfg5():
    ir, sh = "64x0e+64x1o+64x2e", "1x0e+1x1o+1x2e"
    instructions = uvw_instructions(ir, sh, ir)
    return parse_irreps(ir), parse_irreps(sh), parse_irreps(ir), instructions


def test_uvw_path_weights_config5_closed_form():
    in1, in2, out, instructions = _cfg5()
    assert len(instructions) == 11
    assert [sum(1 for ins in instructions if ins[2] == io) for io in range(3)] == [3, 4, 4]
    expected = [CFG5_EXPECTED[ins[2]] for ins in instructions]
    assert uvw_path_weights(in1, in2, out, instructions) == pytest.approx(expected, rel=1e-15)


def test_conv_path_weights_uvw_branch_config5_closed_form():
    from oracle.uvu_conv import path_weights

    in1, in2, out, instructions = _cfg5()
    expected = [CFG5_EXPECTED[ins[2]] for ins in instructions]
    assert path_weights(in1, in2, out, instructions) == pytest.approx(expected, rel=1e-15)


# in1 "2x0e+3x1o" (vars 2, 0.5), in2 "1x0e+2x1o" (vars 3, 0.25), out "4x1o" (var 1.5),
# uvw paths P1 = (0e, 1o) -> 1o with fan 2 * 2 = 4 and P2 = (1o, 0e) -> 1o with fan 3 * 1 = 3:
#   element:   x = 2 * 0.25 * 4 + 0.5 * 3 * 3 = 6.5 for both, alpha = a * 1.5 / 6.5
#   path:      x(P1) = 2 * 0.25 * 4 * 2 = 4, x(P2) = 0.5 * 3 * 3 * 2 = 9
#   component: a = 3; norm: a = d1 * d2 = 3 for both; user weight 0.5 on P2 in the last case.
UVW_VAR_INS = [(0, 1, 0, "uvw", True), (1, 0, 0, "uvw", True)]
UVW_VARS = dict(in1_var=[2.0, 0.5], in2_var=[3.0, 0.25], out_var=[1.5])
UVW_VAR_EXPECTED = {
    ("component", "element"): [math.sqrt(4.5 / 6.5), math.sqrt(4.5 / 6.5)],
    ("component", "path"): [math.sqrt(4.5 / 4), math.sqrt(4.5 / 9)],
    ("norm", "none"): [math.sqrt(4.5), math.sqrt(4.5)],
    ("none", "path"): [math.sqrt(1.5 / 4), math.sqrt(1.5 / 9)],
}


@pytest.mark.parametrize("irrep_norm,path_norm", sorted(UVW_VAR_EXPECTED))
def test_conv_path_weights_uvw_with_variances_closed_form(irrep_norm, path_norm):
    from oracle.uvu_conv import path_weights

    weights = path_weights(parse_irreps("2x0e+3x1o"), parse_irreps("1x0e+2x1o"), parse_irreps("4x1o"),
                           UVW_VAR_INS, irrep_normalization=irrep_norm, path_normalization=path_norm, **UVW_VARS)
    assert weights == pytest.approx(UVW_VAR_EXPECTED[irrep_norm, path_norm], rel=1e-15)


def test_conv_path_weights_uvw_user_weight_closed_form():
    from oracle.uvu_conv import path_weights

    ins = [UVW_VAR_INS[0], UVW_VAR_INS[1] + (0.5,)]
    weights = path_weights(parse_irreps("2x0e+3x1o"), parse_irreps("1x0e+2x1o"), parse_irreps("4x1o"), ins,
                           **UVW_VARS)
    assert weights == pytest.approx([math.sqrt(4.5 / 6.5), math.sqrt(0.5 * 4.5 / 6.5)], rel=1e-15)


def test_uvw_oracle_default_weights_scale_brute_force():
    """The brute force with unit path weights, times the closed-form weight of the
    single path into each output, equals the oracle: "1x0e" x "1x0e" -> "1x0e" has one
    uvw path with fan 1 * 1 (alpha = 1), "2x1o" x "1x0e" -> "3x1o" has fan 2 (alpha 3/2)."""
    for in1, in2, out, alpha in (("1x0e", "1x0e", "1x0e", 1.0), ("2x1o", "1x0e", "3x1o", 1.5)):
        instructions = uvw_instructions(in1, in2, out)
        assert len(instructions) == 1
        a, b, c = parse_irreps(in1), parse_irreps(in2), parse_irreps(out)
        assert uvw_path_weights(a, b, c, instructions) == pytest.approx([math.sqrt(alpha)], rel=1e-15)


@pytest.mark.parametrize("irrep_norm,path_norm", sorted(UVW_VAR_EXPECTED))
def test_package_uvw_normalisation_matches_closed_form(irrep_norm, path_norm):
    from lunaequivariance_amd import TensorProductConfig

    tp = TensorProductConfig("2x0e+3x1o", "1x0e+2x1o", "4x1o", UVW_VAR_INS, shared_weights=True,
                             irrep_normalization=irrep_norm, path_normalization=path_norm, **UVW_VARS)
    assert [i.path_weight for i in tp.instructions] == pytest.approx(UVW_VAR_EXPECTED[irrep_norm, path_norm],
                                                                     rel=1e-14)
