"""Device FArrayBox exchange at the sizes where its two kernels can go wrong:
the smallest boxes that a level takes (five nodes an axis on D3Q39), rows around
the block size, whole blocks, odd extents, ghost widths 0 to 3, both lattices and
storage forms.  Import then export returns the values in storage precision
(exactly in FP64; one FP32 rounding of the deviation in FP32) and leaves ghost
cells alone.  Both population buffers are filled: solid nodes, which no step
writes, hold the imported values in whichever buffer is current."""
import ctypes

import numpy as np
import pytest

from test_gpu_fab import Fab, _hip

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("shape,ghost", [((5, 5, 5), 0), ((5, 5, 5), 3), ((255, 5, 5), 1),
                                         ((257, 5, 5), 0), ((5, 7, 17), 2), ((64, 8, 5), 0),
                                         ((33, 9, 7), 1)])
@pytest.mark.parametrize("lattice", ["d3q27", "d3q39"])
@pytest.mark.parametrize("precision", ["fp32s", "fp64"])
def test_fab_import_export(pkg, orc, lattice, precision, shape, ghost):
    hip = _hip()
    rng = np.random.default_rng(7)
    n = int(np.prod(shape))
    s = pkg.Solver(lattice=lattice, precision=precision)
    if lattice == "d3q39":
        s.set_gas(mach=0.3, shifted=0)
    s.define_level(0, shape)
    fields = {"f": 27} if lattice == "d3q27" else {"f": 39, "g": 39, "lm": 13}
    for name, q in fields.items():
        dense = rng.uniform(0.01, 0.3, (q, n))
        a, b = Fab(hip, shape, q, ghost), Fab(hip, shape, q, ghost)
        a.put(a.with_valid(dense))
        s.import_fab(0, name, a.ptr.value, ghost, a.cstride)
        s.export_fab(0, name, b.ptr.value, ghost, b.cstride)
        out = b.get()
        got = b.valid(out)
        if precision == "fp64" or name == "lm":
            assert np.array_equal(got, dense)
        else:
            # |value - reference| < 0.3 rounded once to FP32: half an ulp
            assert np.abs(got - dense).max() <= 0.3 * 2.0 ** -24
        assert np.isnan(out).sum() == out.size - dense.size
        a.free(), b.free()
    s.close()


@pytest.mark.parametrize("lattice", ["d3q27", "d3q39"])
@pytest.mark.parametrize("precision", ["fp32s", "fp64"])
def test_both_buffers_are_filled(pkg, orc, lattice, precision):
    hip = _hip()
    shape = (32, 24, 16)
    n = int(np.prod(shape))
    s = pkg.Solver(lattice=lattice, precision=precision)
    if lattice == "d3q39":
        s.set_gas(mach=1.5, shifted=1)
    s.define_level(0, shape, periodic=(0, 0, 0))
    s.set_faces(0, [-10] * 6 if lattice == "d3q27" else [-1000, -1000, -11, -6, -1000, -11])
    tri, nrm = pkg.icosphere(4, 4.3, (12.5, 11.75, 7.5), 20260103)
    s.build_links(0, tri, nrm)
    solid = s.download_links(0)[0] == -1001
    assert solid.sum() > 50
    one = np.ones(n)
    if lattice == "d3q27":
        s.init_uniform(0, 1.0, (0.02, 0.0, 0.0))
        dense = {"f": s.download_f(0).reshape(27, n)}
    else:
        s.init_fields(0, one, 1.5 * one, 0 * one, 0 * one, one / 1.4)
        dense = dict(zip(("f", "g"), (v.reshape(39, n) for v in s.download_state(0)[:2])))
    # the solid nodes' values are the test's own, told apart by direction
    for q in dense.values():
        q[:, solid] = 0.01 + 1e-3 * np.arange(len(q))[:, None]
    fabs = {k: Fab(hip, shape, len(v), 1) for k, v in dense.items()}
    for k, fab in fabs.items():
        fab.put(fab.with_valid(dense[k]))
        s.import_fab(0, k, fab.ptr.value, 1, fab.cstride)
    for _ in range(3):
        for k, fab in fabs.items():
            s.export_fab(0, k, fab.ptr.value, 1, fab.cstride)
            got = fab.valid(fab.get())[:, solid]
            assert np.abs(got - dense[k][:, solid]).max() <= (0 if precision == "fp64" else 0.5 * 2.0 ** -24)
        s.step(0, 1)
    for fab in fabs.values():
        fab.free()
    s.close()
