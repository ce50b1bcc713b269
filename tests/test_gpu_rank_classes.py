"""The kernels that a rank's draws run, each set explicitly (a tuning row may
pick another): the group kernel of every rank class against the
one-sample-per-wave kernel (R <= 32) or the block kernel, the block kernel above
R = 64 against the group kernel, and the group kernel that ends the tile
descents.  Indices equal, and in FP64 those of the CPU sampler."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", ["fp64", "fp32"])
@pytest.mark.parametrize("R", [8, 9, 16, 17, 20, 21, 22, 25, 27, 28, 32, 33, 40, 41, 48, 49, 56, 57, 64, 65, 67, 127, 128])
def test_kernels_of_a_rank(oracle, R, precision):
    import fast_tensor_leverage_amd as ftl
    print(f"[gpu] kernels of a rank R={R} {precision}", flush=True)
    rng = np.random.default_rng(R)
    dims = (R + 1, 40 * R + 1, 777)
    U = [rng.standard_normal((n, R)) for n in dims]
    J = 1000
    draws = rng.random(2 * len(dims) * J)
    s = ftl.Sampler(U, J, R, "efficient", precision=precision)
    s.set_option("group_lanes", 0)
    s.set_option("block_threads", 0)
    out = []
    for kernel, tiles in ((0, 0), (1 if R <= 32 else 2 if R <= 64 else 3, 0), (0, 1)):
        s.set_option("draw_kernel", kernel)
        s.set_option("tile_descent", tiles)
        samples = np.zeros((len(dims), J), dtype=np.uint64)
        s.KRPDrawSamples(3, samples, draws)
        out.append(samples)
    np.testing.assert_array_equal(out[0], out[1])
    np.testing.assert_array_equal(out[0], out[2])
    if precision == "fp64":
        ref = oracle.OracleSampler(U, J, R).draw(3, draws)
        np.testing.assert_array_equal(out[0], ref["samples"])
