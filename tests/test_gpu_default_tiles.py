"""The tiles that the nodal walk takes by default against the 16 x 8 tile, which
LGPU_OPT_BRICK_ROWS = 8 selects at every size: no node is missed or done twice,
and FP64 keeps its rounding.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import STATE_FIELDS

pytestmark = pytest.mark.gpu


# k_nodal_block (2, 33), widths 11, 12, 8, 15 and 13 of 256 threads, 16 x 16 (101)
@pytest.mark.parametrize("s", [2, 33, 65, 75, 90, 94, 101, 105])
def test_default_tiles_match_16_by_8(s):
    runs = []
    for rows in (16, 8):
        ctx = la.SedovDevice(s, 11, 1, 1)
        ctx.set_option(la.native.OPT_BRICK_ROWS, rows)
        assert ctx.get_option(la.native.OPT_BRICK_ROWS) == rows
        assert ctx.run(8) == 0
        runs.append({f: ctx.download(f) for f in STATE_FIELDS})
        ctx.close()
    for f in STATE_FIELDS:
        assert np.array_equal(runs[0][f], runs[1][f]), f
