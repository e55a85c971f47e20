"""FP64 RBF evaluation through residues on the INT8 matrix cores
(csrc/rbf_residue.hip) and in the few-column kernel (rbf_thin_kernel) against
long-double products.

Bar, elementwise: the operands are rounded to 2^-62 of the row's 1-norm and
2^-54 of the column's maximum (half a unit each, the scales being powers of
two) and the result once, so
  |Y - ref| <= L1_m max_n (K 2^-62 + 2^-54 + 2^-53) (1 + 2^-20),
L1_m = sum_k |E_mk|, max_n = max_k |X_nk| (|Y| <= L1_m max_n bounds the last
rounding)."""
import numpy as np
import pytest

from conftest import load_inputs, load_orc_rbf, load_surfaces

pytestmark = pytest.mark.gpu

O = load_orc_rbf()


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _bar(E, x):
    K = E.shape[1]
    return (np.abs(x).max(1)[:, None] * np.abs(E).sum(1)[None, :]) * (K * 2.0 ** -62 + 2.0 ** -54 + 2.0 ** -53) * (1 + 2.0 ** -20)


# (M, K, N): tiles of 256 x 128, 64-element chunks, three LDS buffers;
# contractions of more than 550 elements take the residue path
SHAPES = [(1, 551, 65), (255, 575, 65), (256, 576, 127), (257, 577, 128), (300, 640, 129), (513, 641, 200), (40, 705, 256),
          (700, 768, 385), (2000, 320, 400)]
# 32-row blocks of 16-row waves, column tiles of 16 to 64, 32-element chunks
# loaded three ahead; the last is past the work limit of the few-column kernel
THIN = [(1, 1, 1), (15, 31, 3), (31, 32, 16), (33, 33, 17), (129, 95, 48), (64, 97, 49), (300, 129, 64), (257, 550, 65),
        (90, 200, 129), (700, 321, 300)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_residue_products_at_tile_edges(ibm, ctx, shape):
    M, K, N = shape
    rng = np.random.default_rng(M * K + N)
    mats = [rng.standard_normal((M, K + 2)) * 10.0 ** rng.integers(-8, 9, (M, 1)) for _ in range(2)]
    x = rng.standard_normal((N, K)) * 10.0 ** rng.integers(-8, 9, (N, 1))
    mats[1][M // 2] = 0.0                       # a zero row and a zero column
    x[N // 2] = 0.0
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    for j in range(2):
        err = np.abs(Y[j] - O.evaluate(mats[j], K, x))
        assert (err <= _bar(mats[j][:, :K], x)).all(), err.max()
    op.close()


@pytest.mark.parametrize("shape", THIN, ids=lambda s: "x".join(map(str, s)))
def test_thin_products_at_tile_edges(ibm, ctx, shape):
    """Bar: a chain of K fused multiply-adds, K 2^-53 of sum |E||X|."""
    M, K, N = shape
    rng = np.random.default_rng(M * K + N)
    mats = [rng.standard_normal((M, K + 1)) for _ in range(2)]
    x = rng.standard_normal((N, K))
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    for j in range(2):
        scale = np.abs(x) @ np.abs(mats[j][:, :K]).T
        assert (np.abs(Y[j] - O.evaluate(mats[j], K, x)) <= (K + 1) * 2.0 ** -53 * scale).all()
    op.close()


@pytest.mark.parametrize("scale", [1e-300, 1e-160, 1e150, 1e300])
def test_residue_products_at_extreme_scales(ibm, ctx, scale):
    rng = np.random.default_rng(7)
    E, x = rng.standard_normal((200, 600)), rng.standard_normal((70, 600)) * scale
    op = ibm.RbfOperator(ctx, "f64", [_t(E)], 600)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    err = np.abs(Y.cpu().numpy()[0] / scale - O.evaluate(E, 600, x / scale))
    assert (err <= _bar(E, x / scale) + 2.0 ** -52 * np.abs(E).sum(1).max() * 6).all()
    op.close()


def test_residue_error_no_larger_than_a_fused_chain(ibm, ctx):
    """On the RBC operators (value, first and second derivatives) the error
    against long double stays below that of an FP64 fused multiply-add chain
    over the same elements."""
    S, I = load_surfaces(), load_inputs()
    dp, sp = I.bauer_params(600), I.bauer_params(900)
    mats = S.operators(dp, sp, 5, seconds=True)
    rng = np.random.default_rng(3)
    ref = I.rbc_shape(*dp)
    cells = np.stack([I.rotate(ref, 6.0 * rng.random(), rng.standard_normal(3)) + 3.0 * rng.random(3)[:, None]
                      for _ in range(24)], axis=1)
    x = np.ascontiguousarray(cells.reshape(72, -1))
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], 600)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    ld = np.longdouble
    for j, E in enumerate(mats):
        exact = O.evaluate(E, 600, x)
        chain = np.zeros(exact.shape)
        for k in range(600):
            chain = (chain.astype(ld) + x[:, k:k + 1].astype(ld) * E[:, k][None, :].astype(ld)).astype(np.float64)
        a, b = np.linalg.norm((Y[j] - exact).astype(np.float64)), np.linalg.norm((chain - exact).astype(np.float64))
        print(f"operator {j}: residues {a:.3e}, fused chain {b:.3e}")
        assert a <= b
    op.close()


def test_residue_products_carry_nan_and_infinity(ibm, ctx):
    rng = np.random.default_rng(5)
    E, x = np.abs(rng.standard_normal((300, 590))) + 0.1, rng.standard_normal((80, 590))
    x[3, 4], x[66, 0], x[79, 589] = np.nan, np.inf, -np.inf
    op = ibm.RbfOperator(ctx, "f64", [_t(E)], 590)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()[0]
    assert np.isnan(Y[3]).all() and (Y[66] == np.inf).all() and (Y[79] == -np.inf).all()
    fine = [n for n in range(80) if n not in (3, 66, 79)]
    assert (np.abs(Y[fine] - O.evaluate(E, 590, x[fine])) <= _bar(E, x[fine])).all()
    op.close()
    # an operator with a NaN stays on the FP64 matrix cores
    E[10, 10] = np.nan
    op = ibm.RbfOperator(ctx, "f64", [_t(E)], 590)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x[fine])])
    Y = Y.cpu().numpy()[0]
    assert np.isnan(Y[:, 10]).all() and np.isfinite(np.delete(Y, 10, axis=1)).all()
    op.close()


def test_batches_mix_both_paths_and_share_columns(ibm, ctx):
    """Entries of both kernels, and two operators on one
    set of columns, give the values of separate calls."""
    rng = np.random.default_rng(6)
    a = ibm.RbfOperator(ctx, "f64", [_t(rng.standard_normal((300, 600))) for _ in range(2)], 600)
    b = ibm.RbfOperator(ctx, "f64", [_t(rng.standard_normal((90, 600)))], 600)
    wide, thin = _t(rng.standard_normal((100, 600))), _t(rng.standard_normal((12, 600)))
    got = ibm.rbf_eval(ctx, [a, b, a, b], [wide, wide, thin, thin])
    for y, op, x in zip(got, (a, b, a, b), (wide, wide, thin, thin)):
        (alone,) = ibm.rbf_eval(ctx, [op], [x])
        assert np.array_equal(y.cpu().numpy(), alone.cpu().numpy())
    a.close()
    b.close()


def test_captured_tether_step_with_many_cells(ibm, ctx):
    """Tangents evaluated on the solver's second stream inside a captured step
    (24 cells: 72 columns) equal those of the eager step, replay after replay."""
    import torch
    S, I = load_surfaces(), load_inputs()
    ct = S.CellType(I.rbc_shape, 560, 700, 5, I.bauer_params)
    rng = np.random.default_rng(8)
    ref = 0.3 * ct.data_reference()
    x0 = np.stack([ref + 0.4 + 0.8 * rng.random(3)[:, None] for _ in range(24)], axis=1).reshape(-1)
    stream = torch.cuda.Stream()
    gctx = ibm.Context(0, stream=stream)
    runs = []
    with torch.cuda.stream(stream):
        op = ibm.RbfOperator(gctx, "f64", [_t(m) for m in (ct.E, ct.Et, ct.Ep)], ct.nd)
        tether = torch.zeros(3 * 24 * ct.ns, dtype=torch.float64, device="cuda")
        w = _t(ct.w)
        for _ in range(2):
            s = ibm.Solver(gctx, [ibm.periodic(1.6), ibm.dirichlet(1.6), ibm.periodic(1.6)], 16, 1e-4, 10.0, density=1e-3,
                           cell_types=[{"ops": op, "cells": 24, "weights": w, "tether": tether, "stiffness": 1e-3}])
            st = s.zero_state([_t(x0)])
            s.step(st)
            runs.append((s, st))
        (a, sa), (b, sb) = runs
        a.capture(sa)
        for k in range(3):
            a.replay(sa)
            b.step_fixed(sb)
            torch.cuda.synchronize()
            ca, cb = a.cells(0), b.cells(0)
            for key in ("positions", "normals", "sigma", "area", "volume"):
                assert torch.equal(ca[key], cb[key]), (k, key)
            assert torch.equal(sa.xs[0], sb.xs[0])
        for s, _ in runs:
            s.close()
        op.close()
    gctx.close()
