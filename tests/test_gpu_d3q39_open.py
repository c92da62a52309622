"""The periodic D3Q39 step at the boxes where it can go wrong: extents at the
smallest that a level takes (the longest link is 4 on the shifted lattice), whole
blocks and ragged ones; start-up ramps and past them; an iteration cap that
leaves nodes unconverged; multipliers that are no numbers.  FP64 against the oracle: 1e-11 relative (sums of 39
terms through 13 multipliers, 4 steps; measured below 1e-13)."""
import numpy as np
import pytest

from test_gpu_d3q39 import CASES, fields, rel_l2, solver

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape", [(5, 5, 5), (8, 8, 5), (13, 5, 7), (5, 7, 9), (16, 12, 10)])
@pytest.mark.parametrize("step0", [0, 60])
@pytest.mark.parametrize("shifted,mach", CASES)
def test_open_step_by_box(pkg, orc, shifted, mach, step0, shape):
    c = orc.consts39(mach=mach, shifted=shifted)
    f0, g0, lm0 = orc.init39(shape, *fields(shape, mach), c)
    f_o, g_o, lm_o, _, st_o = orc.step_periodic39(shape, f0, g0, lm0, c, step0, 4)
    for prec, tol in (("fp64", 1e-11), ("fp32s", 1e-6)):
        s = solver(pkg, shape, prec, mach, shifted)
        s.upload_state(0, f0, g0, lm0)
        s.set_timestep(0, step0)
        s.step(0, 4)
        f, g, lm = s.download_state(0)
        print(f"{shape} {prec} shifted {shifted}: f {rel_l2(f, f_o):.1e} g {rel_l2(g, g_o):.1e}")
        assert rel_l2(f, f_o) < tol and rel_l2(g, g_o) < tol
        if prec == "fp64":
            assert np.abs(lm - lm_o).max() < 1e-9
            assert s.stats()["newton_iters"] == st_o["lm_iters"]


@pytest.mark.parametrize("shifted,mach", CASES)
def test_unconverged_nodes(pkg, orc, shifted, mach):
    """A cap of one iteration: the nodes that need two are counted and collide
    from the equilibrium of their multipliers, as the general kernel does it."""
    shape = (12, 6, 5)
    c = orc.consts39(mach=mach, shifted=shifted)
    f0, g0, lm0 = orc.init39(shape, *fields(shape, mach), c)
    out = []
    for periodic in ((1, 1, 1), (0, 1, 1)):
        s = pkg.Solver(lattice="d3q39", precision="fp64")
        s.set_gas(mach=mach, shifted=int(shifted), lm_maxit=1)
        s.define_level(0, shape, periodic=periodic)
        if not periodic[0]:
            per = orc.FACE_PERIODIC
            s.set_faces(0, [-1000, per, per, -1000, per, per])
        s.upload_state(0, f0, g0, lm0 + 1e-3)
        s.step(0, 1)
        out.append((s.download_state(0), s.stats()["n_noconv"]))
    assert out[0][1] > 0 and out[1][1] > 0
    # away from the x faces both updates are of the same nodes
    for a, b in zip(out[0][0], out[1][0]):
        a, b = (v.reshape(-1, shape[2], shape[1], shape[0])[..., 4:-4] for v in (a, b))
        assert rel_l2(a, b) < 1e-11


@pytest.mark.parametrize("prec", ["fp64", "fp32s"])
@pytest.mark.parametrize("shifted,mach", CASES)
def test_nan_multipliers_are_reported(pkg, orc, shifted, mach, prec):
    """A NaN among a node's multipliers leaves it without a real alpha root: the
    step says so, with the number of such nodes (one in the first multiplier,
    which stands in every exponent, counts as alpha = 2).  Their new populations
    are NaN, the others as without it."""
    shape = (12, 6, 5)
    n = int(np.prod(shape))
    c = orc.consts39(mach=mach, shifted=shifted)
    f0, g0, lm0 = orc.init39(shape, *fields(shape, mach), c)
    bad = np.arange(7, n, 11)
    lm1 = lm0.reshape(13, n).copy()
    lm1[np.arange(len(bad)) % 13, bad] = np.nan
    first = int((np.arange(len(bad)) % 13 == 0).sum())
    out = []
    for lm in (lm0, lm1.reshape(lm0.shape)):
        s = solver(pkg, shape, prec, mach, shifted)
        s.upload_state(0, f0, g0, lm)
        s.set_timestep(0, 60)
        if lm is lm0:
            s.step(0, 1)
        else:
            with pytest.raises(pkg.UclbsError, match=f": {len(bad) - first} nodes without a real alpha root"):
                s.step(0, 1)
            assert s.stats()["n_trivial"] == first
        out.append(s.download_state(0)[0].reshape(39, n))
    others = np.setdiff1d(np.arange(n), bad)
    assert np.isnan(out[1][:, bad]).all()
    assert np.array_equal(out[0][:, others], out[1][:, others])
