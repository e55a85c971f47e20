"""A large grid whose tiles do not fit the device's free memory is still
spread, by the kernel that needs none."""
import numpy as np
import pytest

from conftest import load_inputs

pytestmark = pytest.mark.gpu


def test_spread_without_memory_for_tiles(ibm):
    import torch
    cells, n = 320, 500                      # 64,000 bricks: 2.6 GB of tiles
    L = cells / 16
    grids = ibm.mac_grids([ibm.periodic(L)] * 3, cells)
    rng = load_inputs().SplitMix64(9)
    x = torch.from_numpy(rng.uniform(3 * n) * L).cuda()
    f = torch.from_numpy(rng.normal(3 * n)).cuda()
    roomy, tight = ibm.Context(0), ibm.Context(0)
    want = ibm.spread(roomy, grids, "cosine", x, f)
    roomy.synchronize()
    roomy.close()
    got = [torch.full_like(w, float("nan")) for w in want]
    torch.cuda.empty_cache()
    free, _ = torch.cuda.mem_get_info()
    taken = torch.empty(free - (2 << 30), dtype=torch.uint8, device="cuda")
    try:
        ibm.spread(tight, grids, "cosine", x, f, out=got)
        tight.synchronize()
    finally:
        del taken
        torch.cuda.empty_cache()
        tight.close()
    for a, b in zip(got, want):
        # both kernels are within 1e-12 of the exact sums (test_gpu_spread_tiles.py)
        assert float((a - b).abs().max()) < 2e-12 * float(b.abs().max())
