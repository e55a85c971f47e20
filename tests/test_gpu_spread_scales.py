"""The spread's fixed-point quantum is a power of two that follows the largest
force, so forces scaled by a power of two give results scaled by it, bit for
bit, down to where the quantum's inverse is still a double."""
import numpy as np
import pytest

from conftest import load_inputs

H = 1 / 16

pytestmark = pytest.mark.gpu


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


@pytest.mark.parametrize("power", [-900, -948, -956, 900])
def test_scaled_forces_give_scaled_results(ibm, ctx, power):
    cells = (16, 16, 16)
    grids = ibm.mac_grids([ibm.periodic(c * H) for c in cells], 16)
    n = 300
    rng = load_inputs().SplitMix64(11)
    x = _t(np.concatenate([rng.uniform(n) * c * H for c in cells]))
    f = 1.0 + rng.uniform(3 * n)
    f[::7] = 0.0
    base = ibm.spread(ctx, grids, "cosine", x, _t(f))
    # the results are 2^10 or so: scaled to stay clear of the subnormals
    scale = 2.0 ** (power - 20 if power < 0 else power)
    got = ibm.spread(ctx, grids, "cosine", x, _t(f * scale))
    ctx.synchronize()
    for a, b in zip(got, base):
        assert np.array_equal(a.cpu().numpy(), b.cpu().numpy() * scale)
