"""Fields read back through the pinned staging: exactly the values that were
set, at the sizes where the copy changes from one piece to several, with
ragged last pieces and shares, and after the staging has grown and been
reused."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu


# bytes per field: 256, just under / at / just over 2 MiB (one piece | four),
# pieces below and at the 8 MiB limit, several rounds of the three slots
@pytest.mark.parametrize("sizes", [[(8, 4)], [(511, 513), (512, 512), (513, 512), (16, 5)], [(1024, 1031), (64, 9)],
                                   [(4096, 2049)]])
def test_fields_come_back_exactly(sizes):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny) for nx, ny in sizes], precision="fp32")
    names = ("rho", "ux", "uy", "cpos", "cneg", "psi")
    data = {}
    for ch, (nx, ny) in enumerate(sizes):
        rng = np.random.default_rng(nx + ny)
        data[ch] = [rng.standard_normal((ny, nx)) for _ in names]
        s.set_fields(ch, *data[ch])
    for ch in list(data) + list(data)[::-1]:  # the staging both grown and already large
        for name, want in zip(names, data[ch]):
            assert np.array_equal(s.get_field(ch, name), want), (sizes[ch], name)
    # the electric field is differentiated from the copied psi
    psi = data[0][-1]
    ex = (np.roll(psi, 1, 1) - np.roll(psi, -1, 1)) * 0.5
    assert np.array_equal(s.get_field(0, "ex"), ex)
