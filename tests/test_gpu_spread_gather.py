"""Few scattered markers on a grid of many bricks: the spread that gathers each
brick's markers (tile_gather_kernel) gives the bits of the tile spread, which
ibm_spread_boxes always takes, and matches the CPU oracle on partial bricks
and beside walls (bar: 1e-12 of the largest value, as for the spread
elsewhere)."""
import numpy as np
import pytest

from conftest import load_inputs

H = 1 / 16

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _domain(ibm, cells, walls=()):
    dom = [(ibm.dirichlet if j in walls else ibm.periodic)(cells[j] * H) for j in range(3)]
    refinement = int(np.gcd.reduce(cells))
    grids = ibm.mac_grids(dom, refinement)
    assert [a.cells for a in grids[0].axis] == list(cells)
    return [(d.length, d.solid, tuple(d.lower), tuple(d.upper)) for d in dom], grids, refinement


def _markers(cells, n, seed):
    rng = load_inputs().SplitMix64(seed)
    x = np.concatenate([rng.uniform(n) * c * H for c in cells])
    return x, rng.normal(3 * n) * 10.0 ** (12 * rng.uniform(3 * n) - 6)       # both conversions to quanta


def _bits(t):
    return t.cpu().numpy().view(np.int64)


# 125 and 240 bricks; 24 and 25 markers of one cell: the most a bin may hold,
# and one too many
@pytest.mark.parametrize("cells", [(40, 40, 40), (48, 40, 64)])
@pytest.mark.parametrize("n,crowd", [(1, 0), (50, 0), (1000, 0), (6000, 0), (60, 24), (60, 25)])
@pytest.mark.parametrize("delta", ["cosine", "peskin", "bspline3"])
def test_gathered_spread_has_the_bits_of_the_tiles(ibm, ctx, cells, n, crowd, delta):
    import torch
    _, grids, _ = _domain(ibm, cells)
    x, f = _markers(cells, n, n + crowd)
    if crowd:
        x = x.reshape(3, n)
        x[:, :crowd] = (np.array([[13.1], [8.2], [39.5]]) + 0.3 * x[:, :crowd] / np.array([[c * H] for c in cells])) * H
        x = x.reshape(-1)
    xd, fd = _t(x), _t(f)
    got = ibm.spread(ctx, grids, delta, xd, fd)
    fixed = [torch.full_like(g, float("nan")) for g in got]
    ibm.spread_sets_noalloc(ctx, grids, delta, [xd], [fd], fixed)
    want = ibm.spread_boxes(ctx, grids, delta, [0, n], xd, fd)
    ctx.synchronize()
    for c in range(3):
        assert np.array_equal(_bits(got[c]), _bits(want[c])) and np.array_equal(_bits(fixed[c]), _bits(want[c])), c


@pytest.mark.parametrize("cells,walls", [((42, 42, 49), ()), ((40, 48, 40), (1,)), ((36, 45, 39), (0, 1, 2)), ((12, 9, 500), ()),
                                         ((4, 48, 512), (1,))])
@pytest.mark.parametrize("n", [2, 700])
def test_gathered_spread_matches_oracle(ibm, orc, ctx, cells, walls, n):
    spec, grids, refinement = _domain(ibm, cells, walls)
    x, f = _markers(cells, n, 17 + n)
    # a third of the markers at the faces of the box, some beyond the walls
    x = x.reshape(3, n)
    for j in range(3):
        k = np.arange(j, n, 9)
        x[j, k] = np.where(k % 2, cells[j] * H, 0.0) + 0.1 * H * (k % 5 - 2)
    x = x.reshape(-1)
    fe = ibm.spread(ctx, grids, "cosine", _t(x), _t(f))
    ctx.synchronize()
    ref = orc.spread(orc.mac_axes(spec, refinement), "cosine", x, f)
    for c in range(3):
        assert np.abs(fe[c].cpu().numpy() - ref[c]).max() < 1e-12 * np.abs(ref[c]).max(), c


def test_a_grid_without_markers_is_zero(ibm, ctx):
    import torch
    _, grids, _ = _domain(ibm, (40, 40, 40))
    out = [torch.full((grids[c].size,), float("nan"), dtype=torch.float64, device="cuda") for c in range(3)]
    empty = torch.empty(0, dtype=torch.float64, device="cuda")
    ibm.spread_sets(ctx, grids, "cosine", [empty], [empty], out=out)
    ctx.synchronize()
    assert all(bool((a == 0).all()) for a in out)
