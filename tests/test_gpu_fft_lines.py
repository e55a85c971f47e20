"""The channel solver's line systems at and beside every chunk length, by the
residual against the CPU oracle's sparse operator.

Bar: max |b - A x| within 1e-13 of (largest row sum of |A|) max |x| + max |b|,
450 units of 2^-52: elimination without pivoting is backward stable on these
diagonally dominant lines, a few units per step of the cyclic reduction, and
the transforms of four points add a few more.
"""
import os

import numpy as np
import pytest

from conftest import ROOT, _load, load_inputs

pytestmark = pytest.mark.gpu

H = 0.05
MAC = [[0.0, 0.5, 0.5], [0.5, 0.0, 0.5], [0.5, 0.5, 0.0]]


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


def _spec(dom):
    return [(d.length, d.solid, tuple(d.lower), tuple(d.upper)) for d in dom]


@pytest.mark.parametrize("ny", [2, 3, 4, 32, 34, 64, 128, 256, 260, 512, 516, 640, 800])
def test_residual_of_every_chunk_length(ibm, orc, ctx, ny):
    fd = _load("orc_fd", os.path.join(ROOT, "oracle", "fd.py"))
    rng = load_inputs().SplitMix64(ny)
    ref = int(np.gcd(ny, 4))

    def check(dom, grid, align, sigma, tau, mean_free):
        A = fd.operator([orc.grid_axes(_spec(dom), ref, align)[j] for j in range(3)], sigma, tau).tocsr()
        b = rng.normal(A.shape[0])
        if mean_free:
            b -= b.mean()
        solver = ibm.FftSolver(ctx, grid)
        x = solver.solve(_t(b), (sigma, tau)).cpu().numpy()
        solver.close()
        bound = abs(A).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max()
        assert np.abs(b - A @ x).max() < 1e-13 * bound, (align, sigma, tau)
        if mean_free:
            assert abs(x.mean()) < 1e-13 * np.abs(x).max()

    dom = [ibm.periodic(4 * H), ibm.dirichlet(ny * H), ibm.periodic(4 * H)]
    grids = ibm.mac_grids(dom, ref)
    for c in (0, 1):                                            # ny and ny - 1 points
        if grids[c].axis[1].points < 2:
            continue
        for tau in (-1e-4, -0.37):
            check(dom, grids[c], MAC[c], 1.0, tau, False)
    pdom = [ibm.periodic(4 * H), ibm.neumann(ny * H), ibm.periodic(4 * H)]
    check(pdom, ibm.centered_grid(pdom, ref), [0.5, 0.5, 0.5], 0.0, 1.0, True)
