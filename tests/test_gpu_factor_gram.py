"""Factor Grams, their reduction and the column norms at the edges of their block
counts (256 and 4,096 rows) and rank tiles, through the low-rank norm and
renormalize_columns."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 7, 8, 16, 17, 32, 33, 48, 49, 64, 65, 128])
@pytest.mark.parametrize("dims", [(1, 2, 3), (255, 257, 256), (4097, 16, 131073)])
def test_norm_and_columns(R, dims):
    import fast_tensor_leverage_amd as ftl
    rng = np.random.default_rng(R + dims[0])
    U = [rng.standard_normal((n, R)) for n in dims]
    lr = ftl.LowRankTensor(R, [u.copy() for u in U])
    G = np.ones((R, R))
    for u in U:
        G = G * (u.T @ u)
    # sums of up to 131,073 rounded products, and N R^2 products of them: the
    # absolute sum bounds the result by cancellation
    bound = np.prod([np.abs(u).T @ np.abs(u) for u in U], axis=0).sum()
    assert abs(lr.get_normsq() - G.sum()) <= 64 * 2.3e-16 * bound
    lr.renormalize_columns(2)
    norm = np.linalg.norm(U[2], axis=0)
    sigma = np.zeros(R)
    lr.get_sigma(sigma)
    np.testing.assert_allclose(sigma, norm, rtol=1e-13)
    np.testing.assert_allclose(lr.U[2], U[2] / norm, rtol=1e-13)
