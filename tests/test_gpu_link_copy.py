"""A link table handed back to the host in pieces: sizes at which the pieces
start (16 MiB), with a whole and with a partial last one, and a small table that
takes the single copy.  What comes back is what was set."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 6, 5), (61, 53, 48), (64, 64, 38), (128, 64, 32), (93, 71, 59)])
def test_table_round_trip(pkg, shape):
    n = int(np.prod(shape))
    rng = np.random.default_rng(n)
    state = rng.integers(-2_000_000, 3, (27, n), dtype=np.int32)
    state[0] = rng.choice([0, 0, 0, -1001], n)
    s = pkg.Solver(precision="fp32s", nu=0.01)
    s.define_level(0, shape)
    s.set_links(0, state)
    for _ in range(2):
        assert np.array_equal(s.download_links(0), state)
