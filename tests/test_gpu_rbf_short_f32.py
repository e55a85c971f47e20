"""FP32 products of short contractions on both sides of the limits of their
128 x 128 tiles (64 elements, 1536 tiles), against FP64 products.

Bar, per value, times sum_k |a_k| |b_k|: FP32 rounds both operands and each of
K additions by at most 2^-24."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [1, 64, 65])
@pytest.mark.parametrize("m,n", [(12165, 1020), (12165, 1025)])          # 96 x 8 and 96 x 9 tiles, two operators
def test_short_products_in_large_and_small_tiles(ibm, ctx, m, n, k):
    import torch
    g = torch.Generator(device="cuda")
    g.manual_seed(k)
    mats = [torch.randn(m, k, dtype=torch.float64, device="cuda", generator=g) for _ in range(2)]
    x = torch.randn(n, k, dtype=torch.float64, device="cuda", generator=g)
    op = ibm.RbfOperator(ctx, "f32", mats, k)
    y = torch.full((2, n, m), float("nan"), dtype=torch.float64, device="cuda")
    ibm.rbf_eval(ctx, [op], [x], ys=[y])
    ctx.synchronize()
    for j in range(2):
        bound = (k + 3) * 2.0 ** -24 * (x.abs() @ mats[j].abs().T)
        assert bool(((y[j] - x @ mats[j].T).abs() <= bound).all()), j
    op.close()
