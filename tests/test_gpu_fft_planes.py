"""The channel solver's plane transforms at all their sizes, beside sizes that
take the separate passes, with vectors at odd 8-byte offsets.

Bar: the residual of the independent stencil, |b - A x| / |b| below 1e-13 (the
solver's bar elsewhere), for the well-conditioned Helmholtz operator of the
timestep.
"""
import pytest

from conftest import load_inputs

pytestmark = pytest.mark.gpu

H = 0.05


@pytest.mark.parametrize("nx", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("nz", [16, 32, 64, 128, 256])
@pytest.mark.parametrize("ny", [4, 64])
def test_residual_at_plane_sizes(ibm, ctx, nx, ny, nz):
    import torch
    dom = [ibm.periodic(nx * H), ibm.dirichlet(ny * H), ibm.periodic(nz * H)]
    grids = ibm.mac_grids(dom, min(nx, ny, nz))
    for c in (1, 2):
        g = grids[c]
        assert g.axis[0].points == nx and g.axis[2].points == nz
        rng = load_inputs().SplitMix64(nx + ny + nz)
        big = torch.from_numpy(rng.normal(g.size + 1)).cuda()
        b, x = big[1:], torch.full_like(big, float("nan"))[1:]
        solver = ibm.FftSolver(ctx, g)
        x = solver.solve(b, (1.0, -5e-4), x=x)
        r = b - ibm.op_apply(ctx, g, (1.0, -5e-4), x)
        assert float(r.norm() / b.norm()) < 1e-13, c
        solver.close()
