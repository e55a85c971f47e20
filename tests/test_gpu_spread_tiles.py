"""The tile spread at the edges of its bricks, chunks and conversions, against
the CPU oracle.

Bar: 1e-12 of the largest value, as for the spread elsewhere.  It holds by
construction: the weights and products carry a few units of 2^-53, and a sum
of m values is off by at most m/2 quanta of at most 2^-61 times the bound
8 m max|f| phi^3 on it (27 m on partly filled bins), below 1e-14 of the sum of
2000 forces of one sign.
"""
import numpy as np
import pytest

from conftest import load_inputs

H = 1 / 16

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _domain(ibm, cells, walls):
    dom = [(ibm.dirichlet if j in walls else ibm.periodic)(cells[j] * H) for j in range(3)]
    refinement = int(np.gcd.reduce(cells))
    grids = ibm.mac_grids(dom, refinement)
    assert [a.cells for a in grids[0].axis] == list(cells)
    return [(d.length, d.solid, tuple(d.lower), tuple(d.upper)) for d in dom], grids, refinement


def _check(ibm, orc, ctx, cells, walls, delta, x, f, split=None):
    import torch
    spec, grids, refinement = _domain(ibm, cells, walls)
    n = len(x) // 3
    parts = [(0, n)] if split is None else [(0, split), (split, n)]
    xs = [_t(x.reshape(3, n)[:, a:b].reshape(-1)) for a, b in parts]
    fs = [_t(f.reshape(3, n)[:, a:b].reshape(-1)) for a, b in parts]
    fe = ibm.spread_sets(ctx, grids, delta, xs, fs)
    fixed = [torch.full_like(r, float("nan")) for r in fe]
    if np.prod(cells) < 2_000_000:                              # what the fixed workspace takes
        ibm.spread_sets_noalloc(ctx, grids, delta, xs, fs, fixed)
    else:
        fixed = fe
    ctx.synchronize()
    ref = orc.spread(orc.mac_axes(spec, refinement), delta, x, f)
    for c in range(3):
        got = fe[c].cpu().numpy()
        assert np.array_equal(got.view(np.int64), fixed[c].cpu().numpy().view(np.int64)), c
        err = np.abs(got - ref[c]).max() / np.abs(ref[c]).max()
        assert err < 1e-12, (c, err)


# periodic axes below, at and beside whole bins (4 cells) and bricks (8 cells),
# alone and beside walls; the last has more bins than one workgroup scans
@pytest.mark.parametrize("cells,walls", [
    ((4, 4, 4), ()), ((5, 7, 9), ()), ((16, 11, 13), ()), ((8, 12, 20), ()), ((25, 32, 17), ()),
    ((9, 7, 5), (1,)), ((12, 4, 7), (0, 2)), ((10, 6, 4), (0, 1, 2)), ((192, 192, 256), (1,)),
])
@pytest.mark.parametrize("delta", ["cosine", "peskin", "bspline3"])
def test_partial_bricks_match_oracle(ibm, orc, ctx, cells, walls, delta):
    n = 777
    rng = load_inputs().SplitMix64(sum(cells))
    x = np.concatenate([rng.uniform(n) * cells[j] * H for j in range(3)])
    f = rng.normal(3 * n) * 10.0 ** (12 * rng.uniform(3 * n) - 6)      # both conversions to quanta
    _check(ibm, orc, ctx, cells, walls, delta, x, f, split=1)


# one brick at and beside a chunk (512 markers), and one stencil origin with
# more markers than the 63 ranks that are told apart
@pytest.mark.parametrize("n", [1, 63, 64, 65, 511, 512, 513, 1500])
@pytest.mark.parametrize("width", [8, 0.25])
def test_crowded_bricks_match_oracle(ibm, orc, ctx, n, width):
    cells = (16, 16, 16)
    rng = load_inputs().SplitMix64(n)
    x = np.concatenate([(4.6 + width * rng.uniform(n)) * H for _ in range(3)])
    f = 1.0 + rng.uniform(3 * n)
    for delta in ("cosine", "peskin"):
        _check(ibm, orc, ctx, cells, (), delta, x, f)


def test_grid_of_many_empty_bricks_keeps_the_brick_kernel(ibm, orc, ctx):
    # 3 x 3 x 850 bricks: more than the fixed workspace holds tiles for
    cells = (17, 17, 6800)
    n = 400
    rng = load_inputs().SplitMix64(5)
    x = np.concatenate([rng.uniform(n) * cells[j] * H for j in range(3)])
    _check(ibm, orc, ctx, cells, (), "cosine", x, rng.normal(3 * n))


@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_non_finite_forces_poison_every_value(ibm, ctx, bad):
    _, grids, _ = _domain(ibm, (9, 12, 16), ())
    rng = load_inputs().SplitMix64(3)
    x = np.concatenate([rng.uniform(100) * c * H for c in (9, 12, 16)])
    f = rng.normal(300)
    f[150] = bad
    fe = ibm.spread(ctx, grids, "cosine", _t(x), _t(f))
    ctx.synchronize()
    assert all(bool(np.isnan(a.cpu().numpy()).all()) for a in fe)
