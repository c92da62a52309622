"""The FP64 root-find at deviations that reach each of its branches: max|x| at
and around the limits of the series of orders 7, 10 and 16 (0.0018, 0.0125,
0.056 at a truncation of 1e-16) and the direct logarithms beyond, alone and
mixed within a wavefront.  One step of a periodic box of noisy populations
against the oracle at the same tolerance 1e-12 on the residual over S2: alpha
within 1e-10 (two residuals of 1e-12 and the rounding of sums of O(x) terms over
S2 ~ x^2, 27 * 2^-53 / x <= 3e-11 at the smallest x = 1e-4), populations within
1e-13."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def noisy(shape, amplitude, seed=5):
    """w_i (1 + amplitude * noise), per node scaled by `amplitude` [n]."""
    import oracle
    n = int(np.prod(shape))
    w = np.asarray(oracle.lattice27()[4])
    r = np.random.default_rng(seed).uniform(-1, 1, (27, n))
    return w[:, None] * (1.0 + amplitude * r)


@pytest.mark.parametrize("amplitude", [1e-4, 1.2e-3, 1.9e-3, 8e-3, 1.4e-2, 0.04, 0.07, 0.3, 0.6])
def test_fp64_alpha_by_deviation(pkg, orc, amplitude):
    shape = (13, 7, 5)
    check(pkg, orc, shape, noisy(shape, amplitude))


def test_fp64_alpha_mixed_wavefronts(pkg, orc):
    shape = (17, 9, 8)
    n = int(np.prod(shape))
    amp = np.random.default_rng(6).choice([1e-4, 1e-3, 5e-3, 0.03, 0.3], n)
    check(pkg, orc, shape, noisy(shape, amp))


def check(pkg, orc, shape, f0):
    nu = 0.01
    f_o, a_o, _ = orc.step_periodic27(shape, f0, 1 / (6 * nu + 1), nsteps=1, tol=1e-12)
    s = pkg.Solver(precision="fp64", nu=nu, alpha_tol=1e-12)
    s.define_level(0, shape)
    s.keep_alpha(True)
    s.upload_f(0, f0)
    s.step(0, 1)
    ea = float(np.abs(s.alpha(0) - np.asarray(a_o).ravel()).max())
    ef = float(np.abs(s.download_f(0).reshape(27, -1) - np.asarray(f_o).reshape(27, -1)).max())
    print(f"alpha diff {ea:.2e}, f diff {ef:.2e}, logarithms at {s.stats()['n_logpath']} nodes")
    assert ea <= 1e-10 and ef <= 1e-13
