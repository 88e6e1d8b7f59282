"""Storage references of narrow rows, a wave each, beside wide ones, a
work-group each: a channel's state over several re-centrings and a restart of
its own does not depend on the channels around it.  The same bits."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu

SIZES = [(320, 6), (10, 13), (256, 5), (4, 70), (257, 9), (65, 8), (130, 7), (512, 4), (64, 11)]


def run(sizes, restart):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=min(4.0, 0.15 * ny)) for nx, ny in sizes], precision="fp32")
    for ch, (nx, ny) in enumerate(sizes):
        g = np.random.default_rng(1000 * nx + ny).standard_normal((5, ny, nx))
        s.set_fields(ch, 1 + 1e-2 * g[0], 1e-2 * g[1], 1e-2 * g[2], 1 + 0.3 * g[3], 1 + 0.3 * g[4])
    s.init_equilibrium()
    s.step(20)  # re-centred at 8 and 16
    if restart is not None:
        s.restart_channel(restart, ekpnp.COLD_NOISE, 3)
        s.step(20)
    s.rebase()
    out = [{sp: s.get_populations(ch, sp) for sp in ("f", "h", "g")} for ch in range(len(sizes))]
    s.close()
    return out


@pytest.mark.parametrize("ch", range(len(SIZES)))
def test_rows_of_one_channel_do_not_depend_on_the_others(ch):
    together, alone = run(SIZES, None)[ch], run([SIZES[ch]], None)[0]
    for sp in together:
        assert np.array_equal(together[sp], alone[sp]), (SIZES[ch], sp)


@pytest.mark.parametrize("ch", [1, 2, 4])
def test_restarted_rows(ch):
    # the cold start's noise is the channel's own: restarted as channel 0 of
    # a context of its own order
    order = [SIZES[ch]] + SIZES[:ch] + SIZES[ch + 1:]
    a, b = run(SIZES, ch), run(order, 0)
    others = [c for c in range(len(SIZES)) if c != ch]
    for i, c in enumerate(others):
        for sp in a[c]:
            assert np.array_equal(a[c][sp], b[1 + i][sp]), (SIZES[c], sp)
