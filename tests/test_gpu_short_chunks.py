"""Node chunks chosen for the shortness of the last one: at most a quarter of
the others' walk.  No node plane is missed or done twice, and FP64 keeps its
rounding.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import STATE_FIELDS

pytestmark = pytest.mark.gpu


# last chunks of 2, 2 and 3 planes after whole ones of 14, 17 and 28
@pytest.mark.parametrize("s", [113, 120, 142])
def test_short_last_chunks_match_chunks_of_nine(s):
    runs = []
    for chunk in (None, 9):
        ctx = la.SedovDevice(s, 11, 1, 1)
        if chunk:
            ctx.set_option(la.native.OPT_BRICK_CHUNK, chunk)
        else:
            whole = ctx.get_option(la.native.OPT_BRICK_CHUNK)
            assert 0 < 4 * ((s + 1) % whole + 1) <= whole + 1
        assert ctx.run(6) == 0
        runs.append({f: ctx.download(f) for f in STATE_FIELDS})
        ctx.close()
    for f in STATE_FIELDS:
        assert np.array_equal(runs[0][f], runs[1][f]), f
