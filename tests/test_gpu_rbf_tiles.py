"""FP32 and split-BF16 products at the edges of both tile sizes, against FP64
products.

Bar, per value, times sum_k |a_k| |b_k|: FP32 rounds both operands and each of
K additions by at most 2^-24; the split drops the low parts' product (2^-16 at
most, as 2^-8 of each) and rounds the low parts (2^-17 each) besides the FP32
sums.
"""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["f32", "bf16x3"])
@pytest.mark.parametrize("m,k", [(3, 3), (63, 64), (64, 65), (65, 31), (129, 300), (200, 1), (4100, 70)])
def test_products_at_tile_edges(ibm, ctx, precision, m, k):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(m + k)
    mats = [torch.randn(m, k, dtype=torch.float64, device="cuda", generator=g) for _ in range(2)]
    op = ibm.RbfOperator(ctx, precision, mats, k)
    rel = (k + 3) * 2.0 ** -24 + (2.0 ** -15 if precision == "bf16x3" else 0.0)
    for n in (1, 63, 64, 65, 128, 130) if m < 4000 else (65, 1030):
        x = torch.randn(n, k, dtype=torch.float64, device="cuda", generator=g)
        y = torch.full((2, n, m), float("nan"), dtype=torch.float64, device="cuda")
        ibm.rbf_eval(ctx, [op], [x], ys=[y])
        ctx.synchronize()
        for j in range(2):
            bound = rel * (x.abs() @ mats[j].abs().T)
            assert bool(((y[j] - x @ mats[j].T).abs() <= bound).all()), (n, j)
    op.close()
