"""computeM's eigensolver on both sides of its size classes (one block with V; A
and the rotations' log with the vectors in a second launch; one or two buffers of
A; odd ranks padded), against NumPy."""
import numpy as np
import pytest

from helpers import gram_pinv

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("R", [1, 2, 3, 4, 5, 16, 31, 32, 33, 34, 63, 64, 65, 95, 96, 97, 98, 127, 128])
@pytest.mark.parametrize("threads", [256, 1024])
def test_compute_m(R, threads):
    import fast_tensor_leverage_amd as ftl
    rng = np.random.default_rng(R)
    U = [rng.standard_normal((n, R)) * np.geomspace(1, 1e-2, R) for n in (900, 2 * R, 517)]
    s = ftl.Sampler(U, 8, R)
    s.set_option("jacobi_threads", threads)
    before = ftl.eigensolver_capped()
    for j in (1, 5):
        modes = [k for k in range(3) if k != j]
        pinv, E = s.compute_m(j)
        ref, G = gram_pinv(U, None if j > 2 else j)
        kept = np.linalg.eigvalsh(G) > 1e-8
        # eigenvalue errors of about R eps |G| and, where the cut leaves a small
        # one, their inverse's amplification
        cond = np.linalg.norm(G, 2) / np.linalg.eigvalsh(G)[kept].min()
        np.testing.assert_allclose(pinv, ref, atol=64 * R * 2.3e-16 * cond * np.linalg.norm(ref, 2))
        for t, k in enumerate(modes):
            P = ref if t + 1 == len(modes) else ref * np.prod([U[q].T @ U[q] for q in modes[t + 1:]], axis=0)
            got = E[k].T @ E[k]
            # a small negative eigenvalue of P is clamped to zero
            np.testing.assert_allclose(got, P, atol=64 * R * 2.3e-16 * cond * np.linalg.norm(P, 2))
            G2 = E[k] @ E[k].T  # orthogonal rows
            np.testing.assert_allclose(G2, np.diag(np.diag(G2)), atol=64 * R * 2.3e-16 * cond * np.abs(G2).max())
    assert ftl.eigensolver_capped() == before


@pytest.mark.parametrize("R", [40, 64])
def test_batched_compute_m(R):
    """Packed requests of a split rank equal the one-shot sampler."""
    import fast_tensor_leverage_amd as ftl
    rng = np.random.default_rng(R)
    srv = ftl.Server(1 << 30, 4)
    sets = [[rng.standard_normal((n, R)) for n in dims] for dims in ((300, 77), (1000, 200, 50), (64, 64, 64, 64))]
    fs = [srv.add_factors(U, 500) for U in sets]
    ids = [srv.submit_on(f, 300 + 50 * i, None if i else 0, 7 + i) for i, f in enumerate(fs)]
    for i, rid in enumerate(ids):
        U = sets[i]
        s = ftl.Sampler(U, 300 + 50 * i, R)
        s.set_seed(7 + i, 0)
        ref = np.zeros((len(U), 300 + 50 * i), dtype=np.uint64)
        s.KRPDrawSamples(len(U) + 1 if i else 0, ref)
        got = srv.wait(rid)
        rows = range(len(U)) if i else range(1, len(U))
        for k in rows:
            np.testing.assert_array_equal(got[k], ref[k])
