"""A seeded draw is a function of its inputs: draws with the default dispatch,
at sizes where they go through the tile kernels, repeat bit for bit.  One
factor with singular values from 1e3 to 2e-4: the mass of a node is a
difference of products up to 1e13 times larger, so a change in the order of a
sum, or of the kernel that evaluates a level, moves indices.  Millions of
samples put many of one bin of the order into one block of the sort."""
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R,J,precision", [(72, 8192, "fp64"), (128, 20_011, "fp32"), (32, 1 << 22, "fp32"),
                                           (24, 1 << 23, "fp64")])
def test_default_draws_repeat(R, J, precision):
    import torch

    import fast_tensor_leverage_amd as ftl
    from fast_tensor_leverage_amd.synth import ill_conditioned_factors
    print(f"[gpu] repeated draws R={R} J={J} {precision}", flush=True)
    dev = torch.device("cuda", 0)
    U, gen = ill_conditioned_factors(torch, 1, 1 << 16, R, dev, seed=R, smin=2e-7)
    given = torch.rand(2 * J, generator=gen, device=dev, dtype=torch.float64)
    s = ftl.Sampler.from_device([1e3 * U[0]], J, R, precision=precision)
    for draws in (None, given):
        first = None
        for _ in range(8):
            samples = torch.zeros((1, J), dtype=torch.int64, device=dev)
            h = torch.empty((J, R), dtype=torch.float64, device=dev)
            w = torch.empty((J,), dtype=torch.float64, device=dev)
            s.set_seed(11, 4)
            s.draw_device(2, samples, h, w, draws)
            torch.cuda.synchronize()
            got = samples, h, w
            first = first or got
            assert [int((a != b).sum()) for a, b in zip(first, got)] == [0, 0, 0]
