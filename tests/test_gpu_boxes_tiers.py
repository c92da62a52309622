"""FP64: a node's update is a function of the node, whatever nodes share its
wavefront.  Periodic boxes of small deviations (most nodes near the limit of the
order-7 series, max|x| of 0.0018) with stray nodes whose neighbours need orders
10, 16 and direct logarithms (0.0125, 0.056 and beyond):
  the same state moved along the axes gives the same alpha and populations, bit
    for bit, moved alike;
  split into uneven boxes (other wavefronts, and ghosts that repeat their source
    node's update) it equals one box bit for bit, with the same iterations."""
import numpy as np
import pytest

from test_gpu_alpha_tiers import noisy
from test_gpu_boxes import _tiling

pytestmark = pytest.mark.gpu
SHAPES = [(64, 48, 40), (17, 13, 9)]


def start(shape):
    n = int(np.prod(shape))
    rng = np.random.default_rng(11)
    amp = rng.uniform(3e-4, 9e-4, n)
    stray = rng.random(n) < 1 / 900
    amp[stray] = rng.choice([5e-3, 0.02, 0.2], stray.sum())
    return noisy(shape, amp, 12)


@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_tiers_moved(pkg, orc, shape):
    grid = shape[::-1]
    f0 = start(shape).reshape(27, *grid)
    out = []
    for move in ((0, 0, 0), (2, 3, 7), (5, 1, 1)):
        s = pkg.Solver(precision="fp64", nu=0.02, alpha_tol=1e-12)
        s.define_level(0, shape)
        s.keep_alpha(True)
        s.upload_f(0, np.roll(f0, move, (1, 2, 3)).reshape(27, -1))
        s.step(0, 1)
        back = [-v for v in move]
        out.append((np.roll(s.alpha(0).reshape(grid), back, (0, 1, 2)),
                    np.roll(s.download_f(0).reshape(27, *grid), back, (1, 2, 3))))
    for a, f in out[1:]:
        print(f"alpha differs by up to {np.abs(a - out[0][0]).max():.1e}")
        assert int((a != out[0][0]).sum()) == 0 and int((f != out[0][1]).sum()) == 0


@pytest.mark.parametrize("shape", SHAPES)
def test_mixed_tiers_by_tiling(pkg, orc, shape):
    f0 = start(shape)
    one = pkg.Solver(precision="fp64", nu=0.02, alpha_tol=1e-12)
    one.define_level(0, shape)
    one.upload_f(0, f0)
    many = pkg.Solver(precision="fp64", nu=0.02, alpha_tol=1e-12)
    many.define_level_boxes(0, _tiling((0, 0, 0), tuple(v - 1 for v in shape), (4, 6, 8, 11), 11))
    many.upload_f(0, many.dense_to_stored(0, f0.reshape(27, *shape[::-1])))
    for steps in (1, 3):
        one.step(0, steps)
        many.step(0, steps)
        a = one.download_f(0).reshape(27, *shape[::-1])
        b = many.stored_to_dense(0, many.download_f(0), shape[::-1])
        assert int((a != b).sum()) == 0
        assert one.stats()["newton_iters"] == many.stats()["newton_iters"]
