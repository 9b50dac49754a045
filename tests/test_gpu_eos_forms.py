"""The fast repeats of k_eos against its general form.

Waves whose elements lie strictly between eosvmin and eosvmax run a form
without those cases; pmin = -0.0 makes every wave take the general form (its
clamp gives the same values up to the sign of zero).  With limits that cut
through the elements' volumes a mesh holds waves of both kinds.
"""
import numpy as np
import pytest

import lulesh_amd as la
from helpers import context_from_oracle, max_rel, upload_state
from oracle_binding import OracleDomain

pytestmark = pytest.mark.gpu

FIELDS = ["e", "p", "q", "ss", "v"]
# FP64 keeps the reference's rounding in both forms; the other two may fuse
# their multiply-adds differently in each (bounds of the forms' own tests)
TOLERANCE = {la.FP64: 0.0, la.FP64_FMA: 1e-11, la.MIXED: 1e-5}


@pytest.mark.parametrize("precision", sorted(TOLERANCE))
@pytest.mark.parametrize("eosvmin,eosvmax", [(1e-9, 1e9), (0.0, 1e9), (1e-9, 1.0), (0.95, 1.01), (0.0, 0.0)])
def test_waves_between_the_volume_limits(precision, eosvmin, eosvmax):
    o = OracleDomain(12, 11, 1, 1)
    for _ in range(40):
        o.call("time_increment")
        assert o.call("lagrange_leapfrog") == 0
    runs = []
    for pmin in (0.0, -0.0):
        k = la.default_constants()
        k.eosvmin, k.eosvmax, k.pmin = eosvmin, eosvmax, pmin
        ctx = context_from_oracle(o, precision=precision, constants=k)
        upload_state(ctx, o)
        dt = o.get("deltatime")
        assert ctx.lagrange_nodal(dt) == 0
        assert ctx.lagrange_elements(dt) == 0
        status, courant, hydro = ctx.time_constraints()
        assert status == 0
        runs.append(({f: ctx.download(f) for f in FIELDS}, courant, hydro))
    (fast, c0, h0), (general, c1, h1) = runs
    for f in FIELDS:
        assert np.all(np.isfinite(fast[f])), f
        assert max_rel(fast[f], general[f]) <= TOLERANCE[precision], f
    assert abs(c0 - c1) <= TOLERANCE[precision] * abs(c1)
    assert h0 == h1


@pytest.mark.parametrize("s,regions,cost", [(1, 1, 0), (2, 11, 1), (5, 21, 4), (17, 11, 0), (50, 21, 2), (102, 21, 2)])
def test_elements_phase_with_shared_and_single_threads(s, regions, cost):
    """Four threads share the repeats of the heaviest elements (here all sizes
    but 1, 2 and 102), or one thread runs them all: the
    FP64 elements phase is the oracle's bit for bit on both sides of the line,
    on partly filled workgroups and with repeat counts below and above the
    count that is shared."""
    o = OracleDomain(s, regions, 2, cost)
    for _ in range(3 if s < 100 else 1):
        o.call("time_increment")
        assert o.call("lagrange_leapfrog") == 0
    o.call("time_increment")
    assert o.call("lagrange_nodal") == 0
    ctx = context_from_oracle(o)
    upload_state(ctx, o)
    assert ctx.lagrange_elements(o.get("deltatime")) == 0
    status, courant, hydro = ctx.time_constraints()
    assert status == 0
    assert o.call("lagrange_elements") == 0
    o.call("calc_time_constraints")
    for f in FIELDS:
        assert np.array_equal(ctx.download(f), o.real(f)), f
    assert (courant, hydro) == (o.get("dtcourant"), o.get("dthydro"))
