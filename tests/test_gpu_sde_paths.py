"""GPU: the SDE kernels' per-path Philox words against the CPU restatement, at
the edges of the path index (its high word enters the second product) and of
the seed."""
import numpy as np
import pytest

from deamd import DE_NOISE_PHILOX, EulerMaruyama, IVP, LinearDiagonal, Milstein, OrnsteinUhlenbeck

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("path_base", [0, (1 << 32) - 70, (1 << 40) + 12345, (1 << 63) - 200])
@pytest.mark.parametrize("dim", [1, 2, 4, 8])
def test_paths_bit_exact(orc, dim, path_base):
    rng = np.random.default_rng([dim, path_base % 997])
    n = 131  # two full wavefronts and a remainder; crosses 2^32 in the second base
    for seed in (1, 0xFFFFFFFF, 0x9E3779B97F4A7C15):
        p = rng.uniform(0.1, 1.5, (dim, 3, n))
        ou = IVP.sde(OrnsteinUhlenbeck(dim, p), 0.0, 0.0315, rng.standard_normal(dim * n),
                     noise=DE_NOISE_PHILOX, seed=seed, path_base=path_base)
        gbm = IVP.sde(LinearDiagonal(dim, p[:, :2].copy()), 0.0, 0.0315,
                      rng.uniform(50.0, 150.0, dim * n), noise=DE_NOISE_PHILOX, seed=seed,
                      path_base=path_base)
        for e in (ou, gbm):
            for method in (EulerMaruyama(1e-3), Milstein(1e-3)):  # a clipped last step
                e.method(method)
                got, want = e.solve(), orc.solve_sde(e)
                assert np.array_equal(got.steps, want.steps)
                assert np.array_equal(got.evals, want.evals)
                assert np.array_equal(got.t, want.t)
                assert np.array_equal(got.y, want.y), (seed, type(method).__name__)
