"""Node sums of the gather path over corner lists of any length.

A hexahedral lattice's nodes have up to eight corners, which k_node reads
together; longer lists go on in a loop, and an empty one gives no force.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import upload_state
from oracle_binding import OracleDomain

pytestmark = pytest.mark.gpu

# sums of at most 16 terms in another grouping: 16 roundings of 2^-53 relative
# to the terms' magnitude, which cancellation can leave far above the sum's
SUM_TOLERANCE = 16 * 2.0 ** -53


def _context(o, starts, corners):
    return la.DeviceContext(
        nodelist=o.ints("nodelist"), lxim=o.ints("lxim"), lxip=o.ints("lxip"), letam=o.ints("letam"),
        letap=o.ints("letap"), lzetam=o.ints("lzetam"), lzetap=o.ints("lzetap"), elemBC=o.ints("elemBC"),
        nodeElemStart=starts, nodeElemCornerList=corners, symmX=o.ints("symmX"), symmY=o.ints("symmY"),
        symmZ=o.ints("symmZ"), regions=o.region_lists(), cost=o.cost, size=o.s, flags=la.native.FLAG_GENERIC)


@pytest.mark.parametrize("extra", [1, 5, 8])
def test_longer_and_empty_corner_lists(extra):
    s = 6
    o = OracleDomain(s, 11, 1, 1)
    for _ in range(30):
        o.call("time_increment")
        assert o.call("lagrange_leapfrog") == 0
    starts, corners = np.array(o.ints("nodeElemStart")), np.array(o.ints("nodeElemCornerList"))
    lists = [corners[a:b] for a, b in zip(starts[:-1], starts[1:])]
    longer, empty = (s + 1) ** 2 + (s + 1) + 1, 2 * (s + 1) ** 2 + 2 * (s + 1) + 2  # interior nodes
    assert len(lists[longer]) == len(lists[empty]) == 8
    changed = list(lists)
    changed[longer] = np.concatenate([lists[longer], lists[longer][:extra]])
    changed[empty] = lists[empty][:0]
    # a third one, which holds just the corners the first has twice
    part = longer + 1
    changed[part] = lists[longer][:extra]
    forces = []
    for each in (lists, changed):
        ctx = _context(o, np.concatenate([[0], np.cumsum([len(v) for v in each])]), np.concatenate(each))
        ctx.set_option(la.native.OPT_KEEP_DIAGNOSTICS, 1)
        upload_state(ctx, o)
        assert ctx.lagrange_nodal(o.get("deltatime")) == 0
        forces.append(np.stack([ctx.download(f) for f in ("fx", "fy", "fz")]))
    plain, got = forces
    others = np.ones(plain.shape[1], bool)
    others[[longer, empty, part]] = False
    assert np.array_equal(got[:, others], plain[:, others])
    assert np.all(got[:, empty] == 0.0)
    scale = np.abs(plain[:, longer]) + np.abs(got[:, part]) + np.abs(plain).max()
    assert np.all(np.abs(got[:, longer] - (plain[:, longer] + got[:, part])) <= SUM_TOLERANCE * scale)
