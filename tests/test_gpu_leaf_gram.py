"""Leaf Grams and the factor copy of the tree build at the edges of their 4 x 4
tiles, thread counts and leaves per block: trees bitwise the oracle's, and a
sampler built from device factors draws as one built from host factors."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# 1-row leaves, trees whose leaves lie on two levels, a last leaf of one row;
# R = 88 and 89 on either side of 256 tiles
@pytest.mark.parametrize("R", [1, 3, 4, 5, 8, 16, 25, 32, 37, 64, 88, 89, 128])
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_device_factors(oracle, R, precision):
    import torch

    import fast_tensor_leverage_amd as ftl
    print(f"[gpu] leaf Grams R={R} {precision}", flush=True)
    rng = np.random.default_rng(R)
    dims = (1, R + 1, 11 * R + 1, 1027, 64 * R)
    U = [rng.standard_normal((n, R)) for n in dims]
    J = 300
    host = ftl.Sampler(U, J, R, "efficient", precision=precision)
    dev = ftl.Sampler.from_device([torch.from_numpy(u).cuda() for u in U], J, R, precision)
    draws = rng.random(2 * len(dims) * J)
    ref = oracle.OracleSampler(U, J, R)
    for k in range(len(dims)):
        np.testing.assert_array_equal(dev.get_tree(k), host.get_tree(k))
        if precision == "fp64":
            np.testing.assert_array_equal(dev.get_tree(k), ref.tree(k))
    a, b = (np.zeros((len(dims), J), dtype=np.uint64) for _ in range(2))
    host.KRPDrawSamples(2, a, draws)
    dev.KRPDrawSamples(2, b, draws)
    np.testing.assert_array_equal(a, b)
