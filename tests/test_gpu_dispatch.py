"""A draw kernel or a cap on its blocks that set_option asks for is the one that
draws, also where draws of that size go through the tile kernels by default.
From one factor with singular values from 1e3 to 2e-4, where node masses are
differences of products up to 1e13 times larger, each kernel draws its own
samples: equal samples mean the same kernel."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,J,options,tiles", [
    (32, 32_768, [], True), (32, 32_768, [("draw_kernel", 1)], False), (32, 32_768, [("grid_blocks", 700)], False),
    (32, 32_768, [("draw_kernel", 1), ("draw_kernel", 0)], True),
    (64, 32_768, [("draw_kernel", 3)], True), (64, 32_768, [("draw_kernel", 2)], False),
    (72, 8192, [("draw_kernel", 2)], True), (72, 8192, [("draw_kernel", 3)], False),
    (72, 8192, [("draw_kernel", 2), ("grid_blocks", 300)], False), (72, 8192, [("block_threads", 128)], True),
])
def test_asked_kernel_draws(R, J, options, tiles):
    import torch

    import fast_tensor_leverage_amd as ftl
    from fast_tensor_leverage_amd.synth import ill_conditioned_factors
    print(f"[gpu] dispatch R={R} J={J} {options}", flush=True)
    dev = torch.device("cuda", 0)
    U, _ = ill_conditioned_factors(torch, 1, 1 << 16, R, dev, seed=R, smin=2e-7)
    s = ftl.Sampler.from_device([1e3 * U[0]], J, R)
    for key, value in options:
        s.set_option(key, value)
    out = {}
    for tile_descent in (2, 0, 1):
        s.set_option("tile_descent", tile_descent)
        s.set_seed(7, 0)
        out[tile_descent] = torch.zeros((1, J), dtype=torch.int64, device=dev)
        s.draw_device(2, out[tile_descent])
    torch.cuda.synchronize()
    assert int((out[0] != out[1]).sum()) > 0
    assert torch.equal(out[2], out[1 if tiles else 0])
