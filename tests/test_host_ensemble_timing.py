"""The launches that an ensemble's kernel timing counts are those it makes: the
kernels of its path once a cycle, and TimeIncrement once a run (later ones are
part of k_dt_reduce).  Host side only, on the fake HIP runtime.
"""
from collections import Counter

import fake_hip


def _timed_run(fake, la, flags, cycles):
    ens = la.Ensemble([5, 9, 7], [1.0] * 3, [1] * 3, [1] * 3, flags=flags)
    ens.set_option(la.native.ENS_OPT_TIMING, 1)
    fake.launches()
    for _ in range(2):
        ens.run(cycles)
    return ens.kernel_stats(), [k.split("<")[0] for k in fake.launches()]


def test_timing_counts_the_launches_made():
    for flags in (0, 1):  # brick path, generic path
        stats, launches = fake_hip.run(_timed_run, flags, 5)
        made = Counter(launches)
        # the timing's names of kernels that have several forms
        names = {"k_nodal_block": "k_nodal_brick", "k_kin_flat": "k_kin_brick",
                 "k_time_increment_ens": "k_time_increment"}
        want = {names.get(k, k): n for k, n in made.items()}
        assert want["k_time_increment"] == 2 and want["k_eos"] > 2
        assert {k: n for k, (n, _) in stats.items() if n} == want
        assert all(ms == n for n, ms in stats.values())  # 1 ms each here
