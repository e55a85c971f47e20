"""A marker at a NaN or infinite position poisons the whole result of a spread
(every value NaN), as a non-finite force does, in each kernel that counts
markers: the tiles of one grid and of a batch of boxes, and the bricks.  Any
finite output would hide a diverged marker."""
import numpy as np
import pytest

from conftest import load_inputs

H = 1 / 16

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _grids(ibm, cells, walls):
    dom = [(ibm.dirichlet if j in walls else ibm.periodic)(cells[j] * H) for j in range(3)]
    return ibm.mac_grids(dom, int(np.gcd.reduce(cells)))


def _markers(cells, n):
    rng = load_inputs().SplitMix64(n)
    return np.concatenate([rng.uniform(n) * c * H for c in cells]), rng.normal(3 * n)


# (17, 17, 6800) has more bricks than the fixed workspace: the brick kernel
@pytest.mark.parametrize("cells,walls", [((9, 12, 16), ()), ((16, 16, 16), (1,)), ((17, 17, 6800), ())])
@pytest.mark.parametrize("bad", [np.nan, np.inf, -np.inf])
def test_non_finite_positions_poison_every_value(ibm, ctx, cells, walls, bad):
    import torch
    grids = _grids(ibm, cells, walls)
    x, f = _markers(cells, 100)
    for axis in range(3):
        at = x.copy()
        at[100 * axis + 37] = bad
        fe = ibm.spread(ctx, grids, "cosine", _t(at), _t(f))
        fixed = [torch.zeros_like(r) for r in fe]
        ibm.spread_sets_noalloc(ctx, grids, "cosine", [_t(at)], [_t(f)], fixed)
        ctx.synchronize()
        assert all(bool(torch.isnan(a).all()) for a in fe + fixed), axis


@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_non_finite_positions_poison_a_batch_of_boxes(ibm, ctx, bad):
    import torch
    grids = _grids(ibm, (16, 16, 16), ())
    x, f = _markers((16, 16, 16), 100)
    x[237] = bad
    fe = ibm.spread_boxes(ctx, grids, "peskin", [0, 40, 40, 100], _t(x), _t(f))
    ctx.synchronize()
    assert all(bool(torch.isnan(a).all()) for a in fe)
