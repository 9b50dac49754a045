"""An ensemble's chunk options set to the value that they read keep the kernels
in use, and bring them back after another value; the autotuner's choice can be
read and set on another ensemble (host side only, on the fake HIP runtime; the
launches name kernels and grids).
"""
import fake_hip


def _ensemble_round_trips(fake, la, sizes, tune):
    n = la.native

    def make():
        ens = la.Ensemble(sizes, [1.0] * len(sizes), [1] * len(sizes), [1] * len(sizes))
        ens.set_option(n.ENS_OPT_GRAPH, 0)
        return ens

    def launches(ens):
        fake.launches()
        ens.run(1)
        return [k for k in fake.launches(grids=True) if "nodal" in k or "kin" in k]

    ens, wrong = make(), []
    choice = ens.autotune(1) if tune else {}
    kernels = launches(ens)
    for option, other in ((n.ENS_OPT_BRICK_CHUNK, 2), (n.ENS_OPT_KIN_CHUNK, 1)):
        value = ens.get_option(option)
        ens.set_option(option, value)
        if launches(ens) != kernels:
            wrong.append(f"option {option} set to its {value}: {launches(ens)}")
        ens.set_option(option, other)
        if launches(ens) == kernels:
            wrong.append(f"option {option} set to {other}: {launches(ens)}")
        ens.set_option(option, value)
        if launches(ens) != kernels or ens.get_option(option) != value:
            wrong.append(f"option {option} back to {value}: {launches(ens)}")
    if tune:  # another ensemble takes the tuner's choice
        again = make()
        for name, option in (("brick_chunk", n.ENS_OPT_BRICK_CHUNK), ("kin_chunk", n.ENS_OPT_KIN_CHUNK),
                             ("nodal_kernel", n.ENS_OPT_NODAL_KERNEL), ("kin_kernel", n.ENS_OPT_KIN_KERNEL)):
            again.set_option(option, choice[name])
        if launches(again) != kernels:
            wrong.append(f"the tuner's {choice} set again: {launches(again)}")
    return kernels, choice, wrong


def test_ensemble_options_set_to_what_they_read_keep_the_kernels():
    """Small bricks and column walks by default, and the autotuner's choice
    (every launch takes as long here, so it is the small-brick kernels), which
    can be read and set on another ensemble."""
    for sizes, tune in (([5, 9, 16, 24], False), (list(range(16, 48)), False), ([5, 9, 16, 24], True),
                        ([118] * 2, True)):
        kernels, choice, wrong = fake_hip.run(_ensemble_round_trips, sizes, tune)
        assert not wrong, (sizes, kernels, wrong)
        if tune:
            assert choice["brick_chunk"] in (4, 6, 8, 11, 16, 22) and choice["kin_chunk"] in (4, 6, 8, 12, 16)
            assert (choice["nodal_kernel"], choice["kin_kernel"]) == (1, 1)
            assert kernels[0].startswith("k_nodal_block") and kernels[1].startswith("k_kin_flat")
