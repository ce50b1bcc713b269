"""Which device factors a tree build reads where they are, and which are copied
first: the rule on the CPU (csrc/factor_source.hpp), and on the GPU factors in
pinned host memory, which are copied."""
import ctypes
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "fast_tensor_leverage_amd", "csrc")

HARNESS = r"""
#include <cstdio>
#include "factor_source.hpp"
int main() {
    // device memory?, owner, base, size; device, address, bytes
    unsigned long long dm, owner, base, size, dev, at, bytes;
    while (std::scanf("%llu %llu %llu %llu %llu %llu %llu", &dm, &owner, &base, &size, &dev, &at, &bytes) == 7)
        std::printf("%d\n", (int)ftl::factor_in_place({dm != 0, (int)owner, base, size}, (int)dev, at, bytes));
}
"""

BASE, SIZE = 0x7f0000000000, 1 << 20
CASES = [
    # device memory, owner, device, address, bytes, read in place
    (1, 0, 0, BASE, SIZE, 1),
    (1, 2, 2, BASE + 4096, SIZE - 4096, 1),
    (1, 0, 0, BASE + SIZE - 8, 8, 1),
    (1, 1, 0, BASE, SIZE, 0),             # another GPU's memory
    (0, 0, 0, BASE, SIZE, 0),             # host, managed or unknown memory
    (1, 0, 0, BASE, SIZE + 8, 0),         # the allocation ends inside the factor
    (1, 0, 0, BASE + 4096, SIZE, 0),
    (1, 0, 0, BASE + SIZE + 8, 8, 0),
    (1, 0, 0, BASE - 8, 16, 0),
    (1, 0, 0, BASE + 4, 8, 0),            # not aligned to its entries
    (1, 0, 0, BASE, (1 << 64) - 8, 0),
]


def test_rule(tmp_path):
    src, exe = tmp_path / "rule.cpp", tmp_path / "rule"
    src.write_text(HARNESS)
    subprocess.run(["g++", "-std=c++17", "-Wall", "-Werror", "-I", CSRC, str(src), "-o", str(exe)], check=True)
    lines = "".join(f"{dm} {own} {BASE} {SIZE} {dev} {at} {n}\n" for dm, own, dev, at, n, _ in CASES)
    out = subprocess.run([str(exe)], input=lines, capture_output=True, text=True, check=True).stdout.split()
    assert [int(x) for x in out] == [c[-1] for c in CASES]


@pytest.mark.gpu
@pytest.mark.parametrize("precision", ["fp64", "fp32"])
def test_pinned_host_factors(precision):
    import torch

    import fast_tensor_leverage_amd as ftl
    from fast_tensor_leverage_amd import _lib
    from fast_tensor_leverage_amd.sampler import PRECISIONS
    print(f"[gpu] factors in pinned host memory {precision}", flush=True)
    rng = np.random.default_rng(3)
    R, J, dims = 24, 500, (1000, 77, 4099)
    U = [torch.from_numpy(rng.standard_normal((n, R))).pin_memory() for n in dims]
    ref = ftl.Sampler([u.numpy() for u in U], J, R, precision=precision)
    L = _lib.load()
    h = ctypes.c_void_p()
    _lib.check(L.ftl_sampler_create_device(3, (ctypes.c_uint64 * 3)(*dims), J, R,
                                           (ctypes.c_void_p * 3)(*[u.data_ptr() for u in U]), PRECISIONS[precision],
                                           ctypes.byref(h)), "create")
    s = ftl.Sampler.__new__(ftl.Sampler)
    s.N, s.J, s.R, s.precision, s.dims, s._matrices, s._h = 3, J, R, precision, list(dims), None, h
    draws = rng.random(2 * 3 * J)

    def compare():
        a, b = (np.zeros((3, J), dtype=np.uint64) for _ in range(2))
        for k in range(3):
            np.testing.assert_array_equal(s.get_tree(k), ref.get_tree(k))
        ref.KRPDrawSamples(4, a, draws)
        s.KRPDrawSamples(4, b, draws)
        np.testing.assert_array_equal(a, b)

    compare()
    new = torch.from_numpy(rng.standard_normal((dims[2], R))).pin_memory()
    ref.update_sampler(2, new.numpy())
    _lib.check(L.ftl_sampler_update_device(h, 2, new.data_ptr()), "update")
    compare()
