"""Matrix-core direct DFT of rows whose width is no power of two: psi against
the oracle at the edges of its 16 x 16 tiles and staged chunks, and mixed with
the other transform families in one context."""
import numpy as np
import pytest

import ekpnp
import oracle as O
from helpers import rel_l2

pytestmark = pytest.mark.gpu


def _fields(nx, ny):
    rng = np.random.default_rng(nx * 131 + ny)
    shp = (ny, nx)
    return (1 + 0.1 * rng.standard_normal(shp), 1 + 0.1 * rng.standard_normal(shp),
            -1 + 0.3 * rng.standard_normal(nx), -0.5 + 0.3 * rng.standard_normal(nx))


def _set(s, ch, nx, ny):
    cp, cn, lo, hi = _fields(nx, ny)
    one, zero = np.ones((ny, nx)), np.zeros((ny, nx))
    s.set_wall_profile(ch, psi_lo=lo, psi_hi=hi)
    s.set_fields(ch, one, zero, zero, cp, cn)


def _want(nx, ny):
    cp, cn, lo, hi = _fields(nx, ny)
    o = O.Oracle(ekpnp.lattice_params(nx, ny), poisson_method=O.POISSON_XDFT_THOMAS)
    o.set_wall_profile(psi_lo=lo, psi_hi=hi)
    o.set_fields(np.ones((ny, nx)), np.zeros((ny, nx)), np.zeros((ny, nx)), cp, cn)
    return o.get_field("psi")


# both sides of the narrow rows' limit and of the two-row-tile widths; nodes,
# modes and rows a multiple of 16, one more and one less; rows shorter than a
# chunk (64, 128 columns; 64 modes), just past it, and the widest
@pytest.mark.parametrize("nx,ny", [(23, 40), (24, 4), (25, 18), (30, 19), (31, 34), (33, 300), (47, 17), (48, 66),
                                   (49, 35), (63, 5), (65, 66), (126, 20), (127, 38), (129, 21), (300, 34), (511, 9),
                                   (1000, 31), (1025, 7), (1999, 8), (2046, 4), (2047, 19)])
def test_psi_matches_oracle(nx, ny):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny)], precision="fp64")
    _set(s, 0, nx, ny)
    want = _want(nx, ny)
    e = rel_l2(s.get_field(0, "psi"), want)
    s.fast_poisson()
    e2 = rel_l2(s.get_field(0, "psi"), want)
    print("dft", nx, ny, e, e2, flush=True)
    assert e < 1e-12 and e2 < 1e-12


def test_mixed_widths_match_single_runs():
    # every transform family in one context (column groups past a channel's
    # last return early), against each channel alone
    sizes = [(64, 40), (100, 43), (1100, 21), (10, 33), (24, 601), (2, 9), (30, 250), (48, 81), (4, 7), (23, 30)]
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny) for nx, ny in sizes], precision="fp64")
    for ch, (nx, ny) in enumerate(sizes):
        _set(s, ch, nx, ny)
    s.fast_poisson()
    for ch, (nx, ny) in enumerate(sizes):
        one = ekpnp.Solver([ekpnp.lattice_params(nx, ny)], precision="fp64")
        _set(one, 0, nx, ny)
        a, b = s.get_field(ch, "psi"), one.get_field(0, "psi")
        print("mixed", nx, ny, rel_l2(a, _want(nx, ny)), flush=True)
        assert np.array_equal(a, b), (nx, ny)
        assert rel_l2(a, _want(nx, ny)) < 1e-12
        one.close()
