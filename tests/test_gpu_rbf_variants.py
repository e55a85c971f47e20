"""The FP64 tile kernels of ibm_rbf_gemm_variant on products that they take:
more than 64 columns, too many blocks for the few-column kernel, and a short
contraction or an operator that keeps no residue planes (with a non-finite
row)."""
import numpy as np
import pytest

from conftest import load_orc_rbf

pytestmark = pytest.mark.gpu

O = load_orc_rbf()


def _t(a):
    import torch
    return torch.from_numpy(np.ascontiguousarray(a)).cuda()


# partial tiles in every direction, whole ones; more than 1024 blocks of 32 x 64
# outputs over the two operators
@pytest.mark.parametrize("shape", [(16385, 33, 65), (8705, 577, 128), (8321, 64, 129), (5505, 40, 300)],
                         ids=lambda s: "x".join(map(str, s)))
@pytest.mark.parametrize("bad", [np.nan, np.inf])
def test_variants_agree_bitwise_and_match_the_oracle(ibm, ctx, shape, bad):
    M, K, N = shape
    rng = np.random.default_rng(M + N)
    mats = [rng.standard_normal((M, K)) for _ in range(2)]
    mats[1][M - 1, K // 2] = bad                       # a spare row
    x = rng.standard_normal((N, K))
    op = ibm.RbfOperator(ctx, "f64", [_t(m) for m in mats], K)
    out = {}
    try:
        for wn in (2, 4, 0):
            ibm.rbf_gemm_variant(wn)
            (Y,) = ibm.rbf_eval(ctx, [op], [_t(x)])
            out[wn] = Y.cpu().numpy()
    finally:
        ibm.rbf_gemm_variant(0)
    assert np.array_equal(out[2], out[4], equal_nan=True) and np.array_equal(out[2], out[0], equal_nan=True)
    assert not np.isfinite(out[2][1][:, M - 1]).any()
    for j in range(2):
        rows = slice(0, M - j)                         # all but the spare row of the second
        scale = np.abs(x) @ np.abs(mats[j][rows]).T
        err = np.abs(out[2][j][:, rows] - O.evaluate(mats[j][rows], K, x))
        assert (err <= (K + 1) * 2.0 ** -53 * scale).all()
    op.close()
