"""lgpu_run's cycle start: a launch of its own, or in the cycle's first kernel
(small bricks, small general meshes).  Either way each cycle's dt comes from
the slots of the cycle before, so a run in pieces of any lengths, host-driven
cycles between them, is the oracle's run.
"""
import numpy as np
import pytest

import lulesh_amd as la
from error_inputs import prepared, qstop, tiny_dt
from helpers import STATE_FIELDS, context_from_oracle, max_rel, upload_state
from oracle_binding import OracleDomain

pytestmark = pytest.mark.gpu

TIMES = ["time", "deltatime", "dtcourant", "dthydro", "cycle"]


def _context(o, form):
    ctx = context_from_oracle(o, generic=form == "generic")
    if form == "walk":  # the cycle start is a launch
        ctx.set_option(la.native.OPT_BRICK_CHUNK, 3)
    if form == "timed":  # waits for the stream instead of the kernels' counts
        ctx.set_option(la.native.OPT_KERNEL_TIMING, 1)
    upload_state(ctx, o)
    return ctx


def _time_state(o):
    ts = la.TimeState()
    for f, _ in ts._fields_:
        v = o.get(f)
        setattr(ts, f, int(v) if f == "cycle" else v)
    return ts


@pytest.mark.parametrize("form", ["block", "walk", "generic", "timed"])
def test_runs_in_pieces_match_the_oracle(form):
    o = OracleDomain(7, 3, 1, 1)
    ctx = _context(o, form)
    ts = _time_state(o)
    for its in (1, 1, 2, 0, 3, 16, 17, 33):  # odd, even, around the 16 that the host runs ahead
        assert o.run(ts.cycle + its) == 0  # both take the last cycle
        assert ctx.run(ts, ts.cycle + its) == 0
        for f in TIMES:  # FP64 keeps the oracle's rounding
            assert getattr(ts, f) == pytest.approx(o.get(f), rel=1e-12, abs=0.0), (its, f)
        # one host-driven cycle between the runs
        assert o.run(ts.cycle + 1) == 0
        assert ctx.lagrange_nodal(o.get("deltatime")) == 0
        assert ctx.lagrange_elements(o.get("deltatime")) == 0
        status, ts.dtcourant, ts.dthydro = ctx.time_constraints()
        assert status == 0
        ts.time, ts.deltatime, ts.cycle = o.get("time"), o.get("deltatime"), int(o.get("cycle"))
    for f in STATE_FIELDS:
        assert max_rel(ctx.download(f), o.real(f)) <= 1e-12, f
    ctx.close()


@pytest.mark.parametrize("form", ["block", "walk", "generic"])
def test_an_error_ends_the_run_at_its_cycle(form):
    o = prepared(tiny_dt, qstop)
    ctx = _context(o, form)
    ts = _time_state(o)
    start = ts.cycle
    assert ctx.run(ts, start + 40) == -2
    assert ts.cycle == start + 1
    ctx.close()
