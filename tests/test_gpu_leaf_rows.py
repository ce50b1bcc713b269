"""Draws at the edges of the rank classes and of the leaf rows' vector loads:
R on either side of 8, 16, 21, 27, 32, 40, 48, 56 and 64, odd and even, with FP64
and FP32 leaves, from factors whose leaves are full, partial and of one row.
Indices equal those of the one-sample-per-wave kernel (R <= 32) or of the
block kernel, and of the CPU sampler in FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("R", [1, 2, 3, 4, 8, 9, 15, 16, 17, 20, 21, 22, 26, 27, 28, 31, 32, 33, 40, 41, 47, 48, 49, 56,
                               57, 63, 64, 65, 67, 127])
def test_rank_classes(oracle, R, precision):
    import fast_tensor_leverage_amd as ftl
    print(f"[gpu] rank classes R={R} {precision}", flush=True)
    rng = np.random.default_rng(R)
    dims = (R + 1, 40 * R + 1, 777)
    U = [rng.standard_normal((n, R)) for n in dims]
    J = 1000
    draws = rng.random(2 * len(dims) * J)
    s = ftl.Sampler(U, J, R, "efficient", precision=precision)
    a, b = (np.zeros((len(dims), J), dtype=np.uint64) for _ in range(2))
    s.KRPDrawSamples(3, a, draws)
    s.set_option("draw_kernel", 1 if R <= 32 else 2)
    s.KRPDrawSamples(3, b, draws)
    np.testing.assert_array_equal(a, b)
    if precision == "fp64":
        ref = oracle.OracleSampler(U, J, R).draw(3, draws)
        np.testing.assert_array_equal(a, ref["samples"])
