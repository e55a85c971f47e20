"""Ranks of scattered markers inside the bins of the tile spread: wavefronts of
64 markers in one bin, in as many bins as are grouped by ballots (24) and in
more, against the CPU oracle (bar: 1e-12 of the largest value)."""
import numpy as np
import pytest

from conftest import load_inputs

H = 1 / 16

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bins", [1, 23, 24, 25, 64])
@pytest.mark.parametrize("n", [64, 1000, 2500])
def test_spread_of_markers_in_many_bins(ibm, orc, ctx, bins, n):
    import torch
    dom = [ibm.periodic(32 * H)] * 3
    grids = ibm.mac_grids(dom, 32)
    rng = load_inputs().SplitMix64(bins + n)
    # marker m in bin (m mod bins) of 4 x 4 x 4 cells
    k = np.arange(n) % bins
    corner = np.stack([4 * (k % 8), 4 * (k // 8 % 8), 4 * ((3 * k) % 8)])
    x = ((corner + 3.9 * rng.uniform(3 * n).reshape(3, n)) * H).reshape(-1)
    f = rng.normal(3 * n)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()  # noqa: E731
    fe = ibm.spread(ctx, grids, "cosine", t(x), t(f))
    ctx.synchronize()
    ref = orc.spread(orc.mac_axes([(d.length, d.solid, tuple(d.lower), tuple(d.upper)) for d in dom], 32), "cosine", x, f)
    for c in range(3):
        assert np.abs(fe[c].cpu().numpy() - ref[c]).max() < 1e-12 * np.abs(ref[c]).max(), c
