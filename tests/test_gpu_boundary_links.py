"""The boundary kernel's link rules one by one: nodes whose link carries each
kind of code -- fluid, halfway, inlet, outlet, freestream, interpolated walls
below, at and above q = 1/2 with and without a fluid node behind, and a code
that names no table -- in tables written by hand, on lists of 1 to 65 nodes
(one wavefront and one node more), against the oracle's step.  FP64: 1e-13.
FP32: 2e-7, two roundings of populations below 1 and of deviations."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CODES = [0, -10, -101, -201, -1000, -1001, -1001 - 250_000_000, -1001 - 499_999_999,
         -1001 - 500_000_000, -1001 - 500_000_001, -1001 - 900_000_000, -50]


@pytest.mark.parametrize("count", [1, 63, 64, 65])
@pytest.mark.parametrize("precision", ["fp64", "fp32s"])
def test_hand_written_links(pkg, orc, precision, count):
    nx, ny, nz = shape = (9, 8, 7)
    n = nx * ny * nz
    rng = np.random.default_rng(count)
    state = np.zeros((27, n), np.int32)
    nodes = rng.choice(n, count, replace=False)
    for k in nodes:
        links = rng.choice(np.arange(1, 27), rng.integers(1, 14), replace=False)
        state[links, k] = rng.choice(CODES[1:], len(links))
    w = orc.lattice27()[4]
    f0 = w[:, None] * (1.0 + 0.02 * rng.uniform(-1, 1, (27, n)))
    nu = 0.01
    states = [(1.0, 0.05, 0.0, 0.01)], [(1.02, 0.0, 0.03, 0.0)], (0.99, 0.02, 0.01, 0.0)
    s = pkg.Solver(precision=precision, nu=nu, alpha_tol=1e-12)
    s.define_level(0, shape, periodic=(1, 1, 1))
    s.set_bc_states(inlets=states[0], outlets=states[1], freestream=states[2])
    s.set_links(0, state)
    s.upload_f(0, f0)
    s.step(0, 1)
    want = orc.step_box27(shape, [orc.FACE_PERIODIC] * 6, state, f0, 1 / (6 * nu + 1), tol=1e-12,
                          inlets=states[0], outlets=states[1], freestream=states[2])[0]
    err = np.abs(s.download_f(0).reshape(27, -1) - np.asarray(want).reshape(27, -1)).max()
    print(f"{precision} {count} nodes: max diff {err:.2e}")
    assert err <= (1e-13 if precision == "fp64" else 2e-7)
