"""Interpolation at the edges of its blocks, on axes shorter than a stencil and
over boxes with few and no markers, against the CPU oracle.

Bar: 1e-12 of the largest value: 64 products of weights that sum to one, each a
few units of 2^-53 off.
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


@pytest.mark.parametrize("cells,walls", [((1, 2, 4), ()), ((2, 1, 1), ()), ((4, 2, 8), (1,)), ((5, 7, 9), ()), ((9, 12, 16), (0, 2)),
                                         ((8, 8, 8), (0, 1, 2))])
@pytest.mark.parametrize("n", [1, 127, 128, 129, 700])
def test_blocks_and_short_axes(ibm, orc, ctx, cells, walls, n):
    spec, grids, refinement = _domain(ibm, cells, walls)
    rng = load_inputs().SplitMix64(n + cells[0])
    # up to a period or a cell beyond the box on either side
    x = np.concatenate([((1 + 2 / cells[j] * (j in walls) + 2 * (j not in walls)) * rng.uniform(n)
                         - (1 / cells[j] if j in walls else 1)) * cells[j] * H for j in range(3)])
    ue = [rng.normal(grids[c].size) for c in range(3)]
    axes = orc.mac_axes(spec, refinement)
    for delta in ("cosine", "peskin", "bspline3"):
        ul = ibm.interpolate(ctx, grids, delta, _t(x), [_t(u) for u in ue]).cpu().numpy()
        ref = orc.interpolate(axes, delta, x, ue)
        assert np.abs(ul - ref).max() <= 1e-12 * max(np.abs(u).max() for u in ue), delta


@pytest.mark.parametrize("counts", [[3], [0, 5, 0, 0, 200, 1, 0], [1] * 63 + [0, 2], [0] * 64 + [70], [2, 0] * 2100 + [300],
                                    [1] * 511, [1] * 512, [1] * 2047, [1] * 2048])
def test_boxes_of_uneven_counts(ibm, orc, ctx, counts):
    cells = (8, 8, 8)
    spec, grids, refinement = _domain(ibm, cells, ())
    off = np.concatenate([[0], np.cumsum(counts)]).astype(int)
    n, nb = int(off[-1]), len(counts)
    rng = load_inputs().SplitMix64(nb)
    x, f = rng.uniform(3 * n) * 8 * H, rng.normal(3 * n)
    one = [rng.normal(grids[c].size) for c in range(3)]
    # box b holds (b + 1) times one field, so the oracle needs one call
    ue = [np.concatenate([(b + 1) * u for b in range(nb)]) for u in one]
    ul = ibm.interpolate_boxes(ctx, grids, "cosine", off.tolist(), _t(x), [_t(u) for u in ue]).cpu().numpy().reshape(3, n)
    axes = orc.mac_axes(spec, refinement)
    ref = orc.interpolate(axes, "cosine", x, one).reshape(3, n) * np.repeat(np.arange(1, nb + 1), counts)
    assert np.abs(ul - ref).max() <= 1e-12 * np.abs(ref).max()
    fe = ibm.spread_boxes(ctx, grids, "cosine", off.tolist(), _t(x), _t(f))
    b = int(np.argmax(counts))
    sl = slice(off[b], off[b + 1])
    ref = orc.spread(axes, "cosine", x.reshape(3, n)[:, sl].reshape(-1), f.reshape(3, n)[:, sl].reshape(-1))
    for c in range(3):
        got = fe[c].cpu().numpy().reshape(nb, -1)[b]
        assert np.abs(got - ref[c]).max() <= 1e-12 * np.abs(ref[c]).max()
