"""k_eos on both sides of the rule that shares the heaviest elements' repeats
between threads (eos_shares): the kernel without sharing, with a group of ten
repeats and the interleaved dispatch order, and the one with it, against the
oracle bit for bit.  Which side a case is on is checked from the kernel that the
host launches for it (no GPU: the fake HIP runtime), so that a change of the
rule cannot move a case without notice.
"""
import numpy as np
import pytest

import fake_hip
import lulesh_amd as la
from helpers import STATE_FIELDS, context_from_oracle, upload_state
from oracle_binding import OracleDomain

FIELDS = ["e", "p", "q", "ss", "v"]
# (s, regions, balance, cost): whether threads share repeats.  11 regions of cost
# 0 have one region of 10 repeats, the others 1
SIDES = {(102, 11, 2, 0): False, (110, 11, 2, 0): False, (1, 1, 1, 0): False, (30, 11, 2, 0): True,
         (102, 21, 2, 2): True}


def _eos_kernel(fake, la, case):
    ctx = la.SedovDevice(*case)
    fake.launches()
    ctx.lagrange_elements(1e-6)
    return fake.launches()[1], ctx.get_option(la.native.OPT_EOS_INTERLEAVE)


@pytest.mark.parametrize("case", sorted(SIDES))
def test_cases_are_on_their_side(case):
    kernel, interleave = fake_hip.run(_eos_kernel, case)
    assert kernel == f"k_eos<PolicyFp64, 256, true, {str(SIDES[case]).lower()}>"
    if case[0] > 100 and not SIDES[case]:
        assert interleave > 0  # the heavy group's workgroups between the others


@pytest.mark.gpu
@pytest.mark.parametrize("case", sorted(SIDES))
def test_elements_phase_matches_the_oracle(case):
    o = OracleDomain(*case)
    for _ in range(3 if case[0] < 100 else 1):
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


@pytest.mark.gpu
def test_dispatch_order_without_sharing_does_not_change_results():
    runs = []
    for k in (None, 0, 1, 4, 7):
        ctx = la.SedovDevice(102, 11, 2, 0)
        if k is not None:
            ctx.set_option(la.native.OPT_EOS_INTERLEAVE, k)
        assert ctx.run(4) == 0
        runs.append(([ctx.download(f) for f in STATE_FIELDS], ctx.ts.dtcourant, ctx.ts.dthydro))
        ctx.close()
    for fields, courant, hydro in runs[1:]:
        assert (courant, hydro) == runs[0][1:]
        for a, b in zip(fields, runs[0][0]):
            assert np.array_equal(a, b)
