"""The order in which a launch takes its samples (option "sample_order") does
not change any output: ordered draws equal unordered ones bitwise."""
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
