"""A link table handed back to the host in pieces: sizes at which the pieces
start (16 MiB), with a whole and with a partial last one, and a small table that
takes the single copy.  What comes back is what was set.  An array that is
pinned already takes the single copy too."""
import ctypes

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(7, 6, 5), (61, 53, 48), (64, 64, 38), (128, 64, 32), (93, 71, 59),
                                   (128, 128, 64)])
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


def test_pinned_destination(pkg):
    n = int(np.prod((64, 64, 38)))
    state = np.random.default_rng(2).integers(-2_000_000, 3, (27, n), dtype=np.int32)
    state[0] = 0
    s = pkg.Solver(precision="fp32s", nu=0.01)
    s.define_level(0, (64, 64, 38))
    s.set_links(0, state)
    pinned = torch.empty((27, n), dtype=torch.int32, pin_memory=True)
    p = ctypes.cast(pinned.data_ptr(), ctypes.POINTER(ctypes.c_int32))
    for _ in range(2):
        pinned.zero_()
        assert s.lib.uclbs_download_links(s.ctx, 0, p, n) == 0
        assert np.array_equal(pinned.numpy(), state)
