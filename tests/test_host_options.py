"""Brick options set to the value that they read keep the kernels, tile and
chunks of the default choice, and bring them back after another value (host
side only, on the fake HIP runtime; the launches name kernels and grids).
"""
import fake_hip


def _round_trips(fake, la, s, precision):
    n = la.native
    ctx = la.SedovDevice(s, precision=precision)

    def launches():
        fake.launches()
        ctx.lagrange_nodal(1e-6)
        ctx.lagrange_elements(1e-6)
        return fake.launches(grids=True)[:2]

    default, wrong = launches(), []
    # another value of each option, which selects or changes the column walks
    for option, other in ((n.OPT_BRICK_CHUNK, 2), (n.OPT_KIN_CHUNK, 1), (n.OPT_BRICK_ROWS, 8)):
        value = ctx.get_option(option)
        ctx.set_option(option, value)
        if launches() != default:
            wrong.append(f"option {option} set to its {value}: {launches()}")
        ctx.set_option(option, other)
        if launches() == default:
            wrong.append(f"option {option} set to {other}: {launches()}")
        ctx.set_option(option, value)
        if launches() != default or ctx.get_option(option) != value:
            wrong.append(f"option {option} back to {value}: {launches()}")
    return default, wrong


def test_options_set_to_what_they_read_keep_the_kernels():
    kernels = set()
    # small bricks, another tile, 16 x 16 with flat kinematics, walks alone
    for s, precision in ((8, 0), (30, 0), (63, 1), (75, 2), (90, 0), (101, 0), (120, 1)):
        default, wrong = fake_hip.run(_round_trips, s, precision)
        assert not wrong, (s, precision, default, wrong)
        kernels |= {k.split("<")[0] + ("<true>" if "true" in k else "") for k in default}
    assert kernels == {"k_nodal_block", "k_nodal_brick", "k_nodal_brick<true>", "k_kin_flat", "k_kin_brick"}
