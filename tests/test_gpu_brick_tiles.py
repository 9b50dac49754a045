"""One problem on the tiles that the nodal walk takes where 16 x 16 threads
would waste columns, and on launches whose last chunks are shorter: the tiles
and chunks change no rounding, and no node is missed or done twice.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import STATE_FIELDS, max_rel

pytestmark = pytest.mark.gpu

# FP64 keeps the reference's rounding on any tile; the other forms may fuse
# multiply-adds differently in each kernel (bounds of the forms' own tests)
TOLERANCE = {la.FP64: 0.0, la.FP64_FMA: 1e-11, la.MIXED: 1e-5}


# widths 11, 12, 8, 15 and 13 of 256 threads; 101 keeps 16
@pytest.mark.parametrize("s,precision", [(65, la.FP64), (75, la.FP64), (90, la.FP64), (94, la.FP64), (101, la.FP64),
                                         (105, la.FP64), (90, la.FP64_FMA), (105, la.MIXED)])
def test_other_tiles_match_16_by_16(s, precision):
    runs = []
    for rows in (None, 16):
        ctx = la.SedovDevice(s, 11, 1, 1, precision=precision)
        if rows:
            ctx.set_option(la.native.OPT_BRICK_ROWS, rows)
            ctx.set_option(la.native.OPT_BRICK_CHUNK, 9)
        assert ctx.get_option(la.native.OPT_BRICK_ROWS) == 16
        assert ctx.run(12) == 0
        runs.append({f: ctx.download(f) for f in STATE_FIELDS})
        ctx.close()
    for f in STATE_FIELDS:
        if precision == la.FP64:
            assert np.array_equal(runs[0][f], runs[1][f]), f
        else:
            assert max_rel(runs[0][f], runs[1][f]) <= TOLERANCE[precision], f
