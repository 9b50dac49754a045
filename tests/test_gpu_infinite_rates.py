"""The hydro constraint of elements whose volume change rate is infinite: its
candidate dvovmax / (|vdov| + 1e-20) (lulesh.cc:2544) is a zero of dvovmax's sign,
below the 1e20 of an element without one, also where no other element of the
workgroup has a candidate.
"""
import numpy as np
import pytest

import lulesh_amd as la

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("precision", [la.FP64, la.FP64_FMA, la.MIXED])
@pytest.mark.parametrize("dvovmax", [0.1, -0.1])
@pytest.mark.parametrize("speed,rate", [(1e308, np.inf), (-1e308, np.inf), (np.nan, np.nan), (0.0, 0.0)])
def test_hydro_constraint_of_one_element(dvovmax, precision, speed, rate):
    k = la.default_constants()
    k.dvovmax = dvovmax
    ctx = la.SedovDevice(1, 1, 1, 1, precision=precision, constants=k)
    xd = np.zeros(8)
    xd[0] = speed
    ctx.upload("xd", xd)
    assert ctx.lagrange_elements(0.0) == 0
    _, _, hydro = ctx.time_constraints()
    vdov = abs(ctx.download("vdov")[0])
    assert np.array_equal(vdov, rate, equal_nan=True)
    want = dvovmax / vdov if np.isinf(vdov) else 1e20
    assert hydro == want and np.signbit(hydro) == np.signbit(want)
    ctx.close()
