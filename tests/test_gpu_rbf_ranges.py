"""FP64 RBF evaluations keep the FP64 chain's componentwise bound whatever the
range of the values in a column or a row, on every path: few columns
(rbf_thin_kernel), residues (rbf_residue.hip) and the columns of an evaluation
by residues that are too wide for them.

Bar, elementwise: a chain of K fused multiply-adds is within K 2^-53 of
sum_k |E_mk||X_nk| (to first order), and one more rounding is allowed for:
  |Y - ref| <= (K + 1) 2^-53 sum |E||X|,
ref being the long-double product (its own error, K 2^-64, is the slack that
the second-order terms need)."""
import numpy as np
import pytest

from conftest import load_inputs, load_orc_rbf, load_surfaces

pytestmark = pytest.mark.gpu

O = load_orc_rbf()


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _check(E, x, Y):
    K = x.shape[1]
    scale = np.abs(x) @ np.abs(E[:, :K]).T
    err = np.abs(Y - O.evaluate(E, K, x))
    worst = (err / np.where(scale > 0, scale, 1.0)).max() * 2.0 ** 53
    assert (err <= (K + 1) * 2.0 ** -53 * scale).all(), f"{worst:.3g} units of 2^-53 of sum |E||X|, K = {K}"


def _narrow(rng, N, K):
    """Values of one binade or two, of either sign: residues throughout."""
    return rng.uniform(0.5, 2.0, (N, K)) * rng.choice([-1.0, 1.0], (N, K)) * 10.0 ** rng.integers(-8, 9, (N, 1))


# (M, K, N): tiles of 256 x 128, 64-element chunks, three LDS buffers
SHAPES = [(1, 551, 65), (255, 575, 65), (256, 576, 127), (257, 577, 128), (300, 640, 129), (513, 641, 200), (40, 705, 256),
          (700, 768, 385), (2000, 320, 400)]


@pytest.mark.parametrize("shape", SHAPES, ids=lambda s: "x".join(map(str, s)))
def test_narrow_columns_at_tile_edges(ibm, ctx, shape):
    M, K, N = shape
    rng = np.random.default_rng(M + K + N)
    mats = [rng.standard_normal((M, K + 2)) * 10.0 ** rng.integers(-8, 9, (M, K + 2)) for _ in range(2)]
    mats[1][M // 2] = 0.0
    x = _narrow(rng, N, K)
    x[N // 2] = 0.0
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    for j in range(2):
        _check(mats[j], x, Y[j])
    op.close()


# both sides of the rule between residues and FP64 products: columns (64),
# contraction (550; 800 where one column tile has many outputs), outputs
@pytest.mark.parametrize("shape", [(300, 600, 64), (300, 600, 65), (300, 550, 70), (300, 551, 70), (3907, 800, 128),
                                   (3907, 801, 128), (3906, 800, 128), (3907, 800, 129)], ids=lambda s: "x".join(map(str, s)))
def test_limits_of_the_residue_path(ibm, ctx, shape):
    M, K, N = shape
    rng = np.random.default_rng(N)
    E, x = rng.standard_normal((M, K)), _narrow(rng, N, K)
    op = ibm.RbfOperator(ctx, "f64", [_t(E)], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    _check(E, x, Y.cpu().numpy()[0])
    op.close()


# FP64 products of more than 64 columns on both sides of 1024 blocks of 32 x 64
# outputs: the few-column kernel and the tiles, in equal bits
@pytest.mark.parametrize("N", [65, 128, 129])
def test_few_column_kernel_and_tiles_give_the_same_bits(ibm, ctx, N):
    M, K = 7000, 90
    rng = np.random.default_rng(N)
    mats = [rng.standard_normal((M, K)) for _ in range(3)]
    x = rng.standard_normal((N, K))
    xd = _t(x)
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)      # 1314 or 1971 blocks
    (Y,) = ibm.rbf_eval(ctx, [op], [xd])
    Y = Y.cpu().numpy()
    op.close()
    for j, E in enumerate(mats):
        _check(E, x, Y[j])
        one = ibm.RbfOperator(ctx, "f64", [_t(E)], K)                # 438 or 657
        (Z,) = ibm.rbf_eval(ctx, [one], [xd])
        assert np.array_equal(Z.cpu().numpy()[0], Y[j])
        one.close()


def _one_hot(rng, M, K):
    E = np.zeros((M, K))
    E[np.arange(M), rng.integers(0, K, M)] = 1.0 + rng.random(M)
    return E


@pytest.mark.parametrize("kind", ["one large entry", "decades", "crossing zero", "zeros", "few zeros", "few tiny",
                                  "alternately huge"])
def test_columns_of_mixed_magnitude(ibm, ctx, kind):
    M, K, N = 300, 600, 100
    rng = np.random.default_rng(len(kind))
    x = rng.standard_normal((N, K))
    if kind == "one large entry":
        x *= 1e-10
        x[np.arange(N), rng.integers(0, K, N)] = 1.0
    elif kind == "decades":
        x *= 10.0 ** rng.integers(-30, 1, (N, K))
    elif kind == "crossing zero":
        x = np.linspace(-1.0, 1.0, K) + 1e-9 * rng.random((N, 1))
    elif kind == "zeros":
        x = np.where(rng.random((N, K)) < 0.5, 0.0, 1.0 + rng.random((N, K)))
    elif kind == "few zeros":
        x = np.where(rng.random((N, K)) < 0.1, 0.0, 1.0 + rng.random((N, K)))
    elif kind == "few tiny":
        x = np.where(rng.random((N, K)) < 0.1, 1e-12, 1.0) * (1.0 + rng.random((N, K)))
    else:
        x[::2] *= 1e17 ** rng.integers(0, 2, (N // 2, K))
    mats = [rng.standard_normal((M, K)), _one_hot(rng, M, K),
            _one_hot(rng, M, K) + 1e-10 * rng.standard_normal((M, K)) * (rng.random((M, K)) < 0.5),
            rng.standard_normal((M, K)) * 10.0 ** rng.integers(-25, 1, (M, K))]
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    for j, E in enumerate(mats):
        _check(E, x, Y[j])
    # every column's value is its own affair: other neighbours, the same bits
    some = x[::3]
    mixed = np.concatenate([_narrow(rng, 30, K), some, _narrow(rng, 40, K)])
    (Z,) = ibm.rbf_eval(ctx, [op], [_t(mixed)])
    assert np.array_equal(Z.cpu().numpy()[:, 30:30 + len(some)], Y[:, ::3])
    op.close()


def test_identity_operator_returns_its_columns(ibm, ctx):
    K, N = 600, 70
    rng = np.random.default_rng(2)
    x = rng.standard_normal((N, K)) * 10.0 ** rng.integers(-18, 1, (N, K))
    op = ibm.RbfOperator(ctx, "f64", [_t(np.eye(K))], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    assert np.array_equal(Y.cpu().numpy()[0], x)
    op.close()


# wide columns among narrow ones: counts at the edges of the FP64 kernels'
# column tiles, and every column
@pytest.mark.parametrize("N,wide", [(65, 1), (129, 31), (200, 32), (200, 33), (200, 63), (200, 64), (200, 65), (300, 128),
                                    (300, 129), (130, 129), (130, 130), (300, 300)])
def test_wide_columns_among_narrow_ones(ibm, ctx, N, wide):
    M, K = 270, 561
    rng = np.random.default_rng(N + wide)
    x = _narrow(rng, N, K)
    which = rng.permutation(N)[:wide]
    x[which] *= 10.0 ** rng.integers(-15, 1, (wide, K))
    mats = [rng.standard_normal((M, K)), _one_hot(rng, M, K)]
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Y = Y.cpu().numpy()
    for j, E in enumerate(mats):
        _check(E, x, Y[j])
    # a column's value does not depend on its neighbours, nor a wide column's
    # on whether it is wide alone
    some = np.sort(np.concatenate([which[:7], rng.permutation(N)[:66]]))
    (Z,) = ibm.rbf_eval(ctx, [op], [_t(x[some])])
    assert np.array_equal(Z.cpu().numpy(), Y[:, some])
    # NaN and infinities in further columns leave the others alone
    x[0, 3], x[N - 1, 560] = np.nan, -np.inf
    (Z,) = ibm.rbf_eval(ctx, [op], [_t(x)])
    Z = Z.cpu().numpy()
    assert np.isnan(Z[0, 0]).all() and not np.isfinite(Z[0, N - 1]).any()
    assert np.array_equal(Z[:, 1:N - 1], Y[:, 1:N - 1])
    op.close()


def test_batch_of_entries_with_and_without_wide_columns(ibm, ctx):
    rng = np.random.default_rng(12)
    shapes = [(300, 600, 90, 5), (520, 640, 150, 0), (40, 700, 200, 200), (90, 600, 90, 70)]
    ops, xs, mats = [], [], []
    for M, K, N, wide in shapes:
        E, x = [rng.standard_normal((M, K)) for _ in range(2)], _narrow(rng, N, K)
        x[:wide] *= 10.0 ** rng.integers(-15, 1, (wide, K))
        ops.append(ibm.RbfOperator(ctx, "f64", [_t(m) for m in E], K))
        mats.append(E)
        xs.append(x)
    dev = [_t(x) for x in xs]
    got = ibm.rbf_eval(ctx, ops + ops[:1], dev + dev[3:])        # the first operator on the last columns too
    for E, x, y in zip(mats + mats[:1], xs + xs[3:], got):
        for j in range(2):
            _check(E[j], x, y.cpu().numpy()[j])
    for op in ops:
        op.close()


def test_captured_tether_step_with_cells_across_a_coordinate_plane(ibm, ctx):
    """Half the cells lie across x = 0 and z = 0, whose coordinates are wide
    columns: tangents on the solver's second stream inside a captured step
    equal those of the eager step, replay after replay."""
    import torch
    S, I = load_surfaces(), load_inputs()
    ct = S.CellType(I.rbc_shape, 560, 700, 5, I.bauer_params)
    rng = np.random.default_rng(8)
    ref = 0.3 * ct.data_reference()
    centres = 0.4 + 0.8 * rng.random((24, 3))
    centres[::2, 0] = 0.02 * rng.random(12)
    centres[::2, 2] = -0.02 * rng.random(12)
    x0 = np.stack([ref + c[:, None] for c in centres], axis=1).reshape(-1)
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
            sites = sa.xs[0].cpu().numpy().reshape(72, -1)
            a.replay(sa)
            b.step_fixed(sb)
            torch.cuda.synchronize()
            ca, cb = a.cells(0), b.cells(0)
            for key in ("positions", "normals", "sigma", "area", "volume"):
                assert torch.equal(ca[key], cb[key]), (k, key)
            assert torch.equal(sa.xs[0], sb.xs[0])
            _check(ct.E, sites, ca["positions"].cpu().numpy().reshape(72, -1))
        for s, _ in runs:
            s.close()
        op.close()
    gctx.close()
