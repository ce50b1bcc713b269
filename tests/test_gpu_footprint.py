"""Device memory of samplers and served requests: at most the trees, factors
and outputs plus a scratch of 3 (R + 1) R doubles per eigensolve and of 2 R + 5
doubles per sample, so that a request that fits a budget goes on fitting it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

ALIGN = 256  # blocks of a server's arena


def _blocks(dims, R, J, sets):
    """Bytes of every block of an FP64 sampler with `sets` computeM buffer sets,
    the factors among them."""
    N = len(dims)
    stride = -(-(R * (R + 1) // 2) // 16) * 16
    rmax = 8
    while rmax < R:
        rmax *= 2
    pad = rmax * (rmax + 1) // 2 + 1088
    out = []
    for n in dims:
        leaves = -(-n // min(R, n))
        out += [8 * n * R, 8 * ((2 * leaves - 1) * stride + pad)]
    out += sets * [8 * R * R, 8 * R * R, 8 * N * R * R, 8 * (N * (2 * R - 1) * stride + pad),
                   8 * (N + 1) * 3 * (R + 1) * R, 8 * (N + 1) * R]
    return out + [8 * J * R, 8 * J * R, 32 * J, 4 * J, 4 * J, 36]


SHAPES = [((1000, 1000, 1000, 1000), 8, 1), ((3000, 40), 16, 2000), ((65536, 70, 64), 25, 2048), ((70, 300, 64), 33, 64), ((500, 40), 40, 1), ((200, 200, 200, 200), 64, 700), ((65, 129, 70), 65, 300),
          ((300, 300, 300), 128, 1000)]


@pytest.mark.parametrize("dims,R,J", SHAPES)
def test_sampler_memory(dims, R, J):
    import fast_tensor_leverage_amd as ftl
    print(f"[gpu] sampler memory {dims} R={R} J={J}", flush=True)
    rng = np.random.default_rng(R)
    s = ftl.Sampler([rng.standard_normal((n, R)) for n in dims], J, R)
    assert s.info()["device_bytes"] <= sum(_blocks(dims, R, J, 2))


@pytest.mark.parametrize("dims,R,J", [s for s in SHAPES if s[1] > 40] + [((70, 300, 64), 33, 4000),
                                                                           ((5000, 3000), 16, 1)])
def test_served_request_fits(dims, R, J):
    import fast_tensor_leverage_amd as ftl
    print(f"[gpu] served request {dims} R={R} J={J}", flush=True)
    up = lambda b: -(-b // ALIGN) * ALIGN
    budget = sum(up(b) for b in _blocks(dims, R, J, 1)) + up(8 * len(dims) * J)
    assert budget >= 1 << 20  # the smallest budget a server takes
    srv = ftl.Server(budget, 1)
    got = srv.wait(srv.submit(list(dims), R, J, None, 5, "fp64"))
    assert all(got[k].max() < n for k, n in enumerate(dims))


def test_order_memory_grows_with_the_options():
    """A sampler whose default takes no order gets the memory for it when an
    option asks, more when a second one does, and draws the same samples."""
    import fast_tensor_leverage_amd as ftl
    print("[gpu] memory of the sample orders", flush=True)
    rng = np.random.default_rng(9)
    dims, R, J = (3001, 1, 517), 12, 3000
    s = ftl.Sampler([rng.standard_normal((n, R)) for n in dims], J, R)
    draws = rng.random(2 * 3 * J)
    out, held = [], []
    for key, value in ((None, 0), ("sample_order", 1), ("tile_descent", 1), ("tile_descent", 0), ("sample_order", 2)):
        if key:
            s.set_option(key, value)
        samples = np.zeros((3, J), dtype=np.uint64)
        s.KRPDrawSamples(4, samples, draws)
        out.append(samples)
        held.append(s.info()["device_bytes"])
    for a in out[1:]:
        np.testing.assert_array_equal(out[0], a)
    assert held[0] < held[1] < held[2] == held[3] == held[4]
