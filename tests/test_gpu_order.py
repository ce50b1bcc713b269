"""The order in which a launch takes its samples (option "sample_order") does
not change any output: ordered draws equal unordered ones bitwise.  Descents in
tiles (option "tile_descent") draw the same samples."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _draw(s, N, J, R, j, draws):
    samples, h, w = np.zeros((N, J), dtype=np.uint64), np.zeros((J, R)), np.zeros(J)
    s.set_seed(5, 3)
    s.KRPDrawSamples_materialize(j, samples, h, w, draws)
    return samples, h, w


# one sample, partial waves and blocks, more samples than one block's counts;
# every draw kernel (groups, one sample per wave, one per block); one-row modes
@pytest.mark.parametrize("R,J,precision,options", [
    (3, 1, "fp64", {}), (8, 7, "fp64", {}), (16, 65, "fp32", {}), (32, 257, "fp64", {}), (32, 4099, "fp32", {}),
    (25, 1023, "fp64", {"draw_kernel": 1}), (64, 130, "fp64", {}), (100, 515, "fp32", {}), (128, 9, "fp64", {}),
    (32, 1000, "fp64", {"mode_split": 0}), (16, 300, "fp64", {"grid_blocks": 3}),
])
@pytest.mark.parametrize("given", [True, False])
def test_ordered_draws_equal_unordered(R, J, precision, options, given):
    import fast_tensor_leverage_amd as ftl
    rng = np.random.default_rng(R * 1000 + J)
    U = [rng.standard_normal((n, R)) for n in (3001, 1, 517)]
    draws = rng.random(2 * 3 * J) if given else None
    if given:
        draws[:2] = 0.0, 1.0 - 2.0 ** -53
    s = ftl.Sampler(U, J, R, precision=precision)
    for k, v in options.items():
        s.set_option(k, v)
    for j in (1, 4):
        out = {}
        for order in (0, 1, 1):
            s.set_option("sample_order", order)
            out.setdefault(order, []).append(_draw(s, 3, J, R, j, draws))
        for got in out[1]:
            for a, b in zip(out[0][0], got):
                np.testing.assert_array_equal(a, b)


# every rank block (16 columns) on both sides of its edge; partial tiles (16
# samples) and blocks (64); modes of one row, fewer rows than R, a partial bottom
# level and one whose FP32 levels start inside the tile descent
@pytest.mark.parametrize("R", [1, 15, 16, 17, 32, 33, 48, 63, 64, 65, 80, 81, 96, 97, 112, 113, 128])
@pytest.mark.parametrize("J,precision", [(1, "fp64"), (15, "fp32"), (17, "fp64"), (64, "fp32"), (1025, "fp64"),
                                         (999, "fp32")])
def test_tile_descents_equal_group_descents(R, J, precision):
    import fast_tensor_leverage_amd as ftl
    rng = np.random.default_rng(R * 1000 + J)
    dims = (40 * R + 5, 1, 7, 13 * R)
    U = [rng.standard_normal((n, R)) for n in dims]
    s = ftl.Sampler(U, J, R, precision=precision)
    draws = rng.random(2 * len(dims) * J)
    for j, d in ((0, draws), (5, None), (2, draws)):
        out = []
        for tiles in (0, 1, 1):
            s.set_option("sample_order", 0)
            s.set_option("tile_descent", tiles)
            out.append(_draw(s, len(dims), J, R, j, d))
        # the node masses differ in their last bits only: a sample moves when
        # its uniform is within about 1e-15 of a boundary of the 128 x 40 rows
        np.testing.assert_array_equal(out[0][0], out[1][0])
        np.testing.assert_array_equal(out[0][1], out[1][1])
        np.testing.assert_allclose(out[1][2], out[0][2], rtol=1e-12)
        for a, b in zip(out[1], out[2]):
            np.testing.assert_array_equal(a, b)


def test_tile_descents_against_oracle(oracle):
    import fast_tensor_leverage_amd as ftl
    R, J, dims = 72, 300, (1000, 333, 90)
    rng = np.random.default_rng(8)
    U = [rng.standard_normal((n, R)) for n in dims]
    draws = rng.random(2 * 3 * J)
    s = ftl.Sampler(U, J, R)
    s.set_option("tile_descent", 1)
    samples, h, w = _draw(s, 3, J, R, 4, draws)
    ref = oracle.OracleSampler(U, J, R).draw(4, draws)
    sure = ref["margins"] > 1e-10
    assert np.array_equal(samples[:, sure], ref["samples"][:, sure])
    agree = np.all(samples == ref["samples"], axis=0)
    np.testing.assert_allclose(w[agree], ref["weights"][agree], rtol=1e-10)
