"""Device FArrayBox exchange at the sizes where its two kernels can go wrong:
the smallest boxes that a level takes (five nodes an axis on D3Q39), rows around
the block size, whole blocks, odd extents, ghost widths 0 to 3, both lattices and storage forms.  Import then export returns the values
in storage precision (exactly in FP64; one FP32 rounding of the deviation in
FP32), leaves ghost cells alone, and fills both population buffers (a step
reads one and a download of the next reads the other)."""
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
