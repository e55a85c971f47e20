"""The channel solver on lines of few rows (64 modes a block up to 8 rows) with
full and partial blocks of modes, by the residual against the CPU oracle's
sparse operator.

Bar: max |b - A x| within 1e-13 of (largest row sum of |A|) max |x| + max |b|
times the transforms' depth, log2 of 256 x 16 points: elimination is backward
stable on these diagonally dominant lines and a radix-2 transform adds a few
units of 2^-52 a stage, of which the bar has 450 for one."""
import os

import numpy as np
import pytest

from conftest import ROOT, _load, load_inputs

pytestmark = pytest.mark.gpu

H = 1 / 16


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("nx", [4, 128, 256])
@pytest.mark.parametrize("ny", [2, 4, 6, 8, 10])
def test_residual_of_short_lines(ibm, orc, ctx, nx, ny):
    fd = _load("orc_fd", os.path.join(ROOT, "oracle", "fd.py"))
    rng = load_inputs().SplitMix64(nx + ny)
    nz, ref = 16, int(np.gcd.reduce([nx, ny, 16]))
    for wall, sigma, tau in ((ibm.dirichlet, 1.0, -0.37), (ibm.neumann, 0.0, 1.0)):
        dom = [ibm.periodic(nx * H), wall(ny * H), ibm.periodic(nz * H)]
        grid = ibm.centered_grid(dom, ref)
        assert [a.points for a in grid.axis] == [nx, ny, nz]
        spec = [(d.length, d.solid, tuple(d.lower), tuple(d.upper)) for d in dom]
        A = fd.operator([orc.grid_axes(spec, ref, [0.5, 0.5, 0.5])[j] for j in range(3)], sigma, tau).tocsr()
        b = rng.normal(A.shape[0])
        if sigma == 0:
            b -= b.mean()
        solver = ibm.FftSolver(ctx, grid)
        x = solver.solve(_t(b), (sigma, tau)).cpu().numpy()
        solver.close()
        bound = abs(A).sum(axis=1).max() * np.abs(x).max() + np.abs(b).max()
        assert np.abs(b - A @ x).max() < 1e-13 * np.log2(nx * nz) * bound, (sigma, tau)
