"""An ensemble whose kernels or chunks cannot be changed, because the device has
no memory for the new tables, keeps the ones it has: what it launches next is
made for the tables that it reads (host side only, on the fake HIP runtime,
which marks launches on freed tables or on those of another kernel).
"""
import fake_hip


def _refused_change(fake, la, option, value):
    n = 31  # column walks of several planes by default, whose chunks of one take larger tables
    ens = la.Ensemble(list(range(10, 10 + n)), [1.0] * n, [1] * n, [1] * n)
    ens.set_option(la.native.ENS_OPT_GRAPH, 0)
    seen = []
    for _ in range(2):
        fake.launches()
        ens.run(1)
        seen.append([k for k in fake.launches() if "nodal" in k or "kin" in k])
        if len(seen) == 1:
            fake.fail_malloc_after(0)
            try:
                ens.set_option(option, value)
                raise SystemExit("accepted")
            except RuntimeError as e:
                assert "ENOMEM" in str(e)
            fake.fail_malloc_after(-1)
    return seen


def test_a_refused_chunk_keeps_the_tables():
    for option in (7, 8):  # ENS_OPT_BRICK_CHUNK, ENS_OPT_KIN_CHUNK
        before, after = fake_hip.run(_refused_change, option, 1)
        assert before == after and not any("!" in k for k in after), after


def _failing_autotune(fake, la, mallocs):
    n = 31
    ens = la.Ensemble(list(range(10, 10 + n)), [1.0] * n, [1] * n, [1] * n)
    ens.set_option(la.native.ENS_OPT_GRAPH, 0)
    fake.fail_malloc_after(mallocs)
    try:
        ens.autotune(1)
        raise SystemExit("accepted")
    except RuntimeError as e:
        assert "ENOMEM" in str(e)
    fake.fail_malloc_after(-1)
    fake.launches()
    ens.run(1)
    return fake.launches()


def test_an_autotune_that_fails_leaves_kernels_with_their_tables():
    # the snapshot, then the tables of one candidate after the other
    for mallocs in (1, 2, 3):
        launches = fake_hip.run(_failing_autotune, mallocs)
        assert not any("!" in k for k in launches), (mallocs, launches)
