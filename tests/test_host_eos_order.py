"""The order in which k_eos's workgroups are dispatched, from the table that it
reads: the workgroups cover the work list once, and their order is the rule's
restated here from the region runs, for both constructors (host side only, on the
fake HIP runtime).
"""
import fake_hip


def _orders(fake, la, s, regions, balance, cost, precision, interleaves, host):
    n = la.native
    if host:
        owner = la.HostDomain(s, regions, balance, cost)
        owner.attach_device(precision)
        ptr = owner.device()
    else:
        owner = la.SedovDevice(s, regions, balance, cost, precision=precision)
        ptr = owner.ptr
    import ctypes
    lib, out = la.gpu_lib(), []
    for k in interleaves:
        if k is not None:
            la.check(lib.lgpu_set_option(ptr, n.OPT_EOS_INTERLEAVE, k))
        v = ctypes.c_int64()
        la.check(lib.lgpu_get_option(ptr, n.OPT_EOS_INTERLEAVE, ctypes.byref(v)))
        la.check(lib.lgpu_lagrange_elements(ptr, 1e-6))
        out.append([v.value, fake.eos_slots()])
    runs = [a.tolist() for a in la.region_runs(s, regions, balance)]
    return out, runs


def _rep(r, regions, cost):  # lulesh.cc:2390-2400, r from 0
    return 1 if r < regions // 2 else 1 + cost if r < regions - (regions + 15) // 20 else 10 * (1 + cost)


def _expected(slots, k, perm, mixed):
    """The slots in the order of interleave k."""
    by_list = sorted(slots)  # work-list order
    if k == 0:
        return by_list
    top = by_list[0][2]
    heavy = [s for s in by_list if s[2] == top]
    rest = sorted((s for s in by_list if s[2] != top), key=lambda s: perm[s[0]])
    if not mixed:
        heavy, rest = heavy[::-1], rest[::-1]
    order = []
    while heavy or rest:
        order += heavy[:1] + rest[:k]
        heavy, rest = heavy[1:], rest[k:]
    return order


def test_dispatch_order():
    interleaves = [None, 0, 1, 4, 7]
    for case in ((1, 1, 1, 1, 0), (30, 11, 1, 1, 0), (61, 21, 2, 2, 1), (64, 5, 1, 0, 0), (64, 11, 1, 1, 2),
                 (80, 16, 3, 4, 1), (90, 11, 2, 0, 0)):
        s, regions, balance, cost, precision = case
        for host in (False, True):
            if host and s > 64:
                continue
            orders, (reg, length) = fake_hip.run(_orders, *case, interleaves, host)
            groups, at = {}, 0
            for r, n in zip(reg, length):
                groups.setdefault(_rep(r - 1, regions, cost), []).extend(range(at, at + n))
                at += n
            perm = [e for rep in sorted(groups, reverse=True) for e in groups[rep]]
            rep_at = [rep for rep in sorted(groups, reverse=True) for _ in groups[rep]]
            for k, slots in orders:
                slots = [tuple(x) for x in slots]
                covered = [p for pos, count, rep, _ in sorted(slots) for p in range(pos, pos + count)]
                assert covered == list(range(s ** 3)), case
                assert all(rep_at[pos] == rep == rep_at[pos + count - 1] for pos, count, rep, _ in slots), case
                assert slots == _expected(slots, k, perm, precision == 1), (case, host, k)
