"""The small-brick kernels (k_nodal_block, k_kin_flat) against the others.

Small bricks run the nodal pass in blocks of elements and the kinematics on
consecutive elements; setting a chunk selects the kernels that walk up
columns, and LGPU_FLAG_GENERIC the gathers.  All of them add corners in the
reference's order and evaluate the same formulas.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import STATE_FIELDS, context_from_oracle, max_rel, upload_state
from oracle_binding import OracleDomain

pytestmark = pytest.mark.gpu

# FP64 keeps the reference's rounding in every kernel; the other forms may
# fuse multiply-adds differently in each (bounds of the forms' own tests)
TOLERANCE = {la.FP64: 0.0, la.FP64_FMA: 1e-11, la.MIXED: 1e-5}
NODE_DIAGNOSTICS = ["fx", "fy", "fz", "xdd", "ydd", "zdd"]


# block edges: one node more and less than whole blocks, single elements
@pytest.mark.parametrize("s,precision", [(s, la.FP64) for s in (1, 2, 3, 5, 6, 9, 13, 16, 30, 46)] +
                         [(s, p) for s in (2, 13, 30) for p in (la.FP64_FMA, la.MIXED)])
def test_small_brick_kernels_match_the_others(s, precision):
    o = OracleDomain(s, 11, 1, 1)
    small, walk, generic = (context_from_oracle(o, precision=precision, generic=g) for g in (False, False, True))
    walk.set_option(la.native.OPT_BRICK_CHUNK, 3)
    walk.set_option(la.native.OPT_KIN_CHUNK, 2)
    ctxs = (small, walk, generic)
    for ctx in ctxs:
        upload_state(ctx, o)
        ctx.set_option(la.native.OPT_KEEP_DIAGNOSTICS, 1)
    dt = o.get("deltatime")
    for _ in range(8):
        constraints = []
        for ctx in ctxs:
            assert ctx.lagrange_nodal(dt) == 0
            assert ctx.lagrange_elements(dt) == 0
            status, c, h = ctx.time_constraints()
            assert status == 0
            constraints.append((c, h))
        tol = TOLERANCE[precision]
        for c, h in constraints[1:]:
            assert abs(c - constraints[0][0]) <= tol * c and abs(h - constraints[0][1]) <= tol * h
        dt = min(constraints[0][0] / 2, 1.1 * dt)
    for f in STATE_FIELDS + NODE_DIAGNOSTICS:
        got = small.download(f)
        for ctx in (walk, generic):
            assert max_rel(got, ctx.download(f)) <= tol, f


def test_small_brick_device_loop_ends_like_the_walk():
    """lgpu_run past the stop time: the cycles enqueued after the loop's end
    carry the state over unchanged in both nodal kernels."""
    runs = []
    for chunk in (None, 3):
        d = la.SedovDevice(6)
        if chunk:
            d.set_option(la.native.OPT_BRICK_CHUNK, chunk)
        assert d.run(10 ** 6) == 0
        runs.append((d.ts.cycle, [d.download(f) for f in STATE_FIELDS]))
    assert runs[0][0] == runs[1][0] > 0
    for a, b in zip(runs[0][1], runs[1][1]):
        assert np.array_equal(a, b)
