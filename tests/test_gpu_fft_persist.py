"""The pipelined x-transforms' two prefetch depths (tiles of up to 1024 and of
up to 2048 values): the same psi, bit for bit, in batches of mixed widths with
more tiles than work-groups, ragged last tiles and rows of a tile each."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes", [[(8, 300), (16, 65), (32, 33), (64, 64)] * 3, [(128, 18), (256, 9), (512, 5), (1024, 7)],
                                   [(2048, 6)], [(2048, 2000), (8, 9)]])
def test_prefetch_depths_agree(sizes):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=min(4.0, 0.15 * ny)) for nx, ny in sizes], precision="fp32")
    for ch, (nx, ny) in enumerate(sizes):
        rng = np.random.default_rng(10 * nx + ny + ch)
        z = rng.standard_normal(nx)
        s.set_wall_profile(ch, psi_lo=z, psi_hi=z[::-1].copy())
        one, zero = np.ones((ny, nx)), np.zeros((ny, nx))
        s.set_fields(ch, one, zero, zero, 1 + 0.3 * rng.standard_normal((ny, nx)), 1 + 0.3 * rng.standard_normal((ny, nx)))
    s.init_equilibrium()
    s.stream_collide_save()
    got = []
    for elems in (1024, 2048, 1024):
        s.set_poisson_plan(elems, 16, 1)
        assert s.poisson_plan()["fft_kernels"] == "persistent"
        s.fast_poisson()
        got.append([s.get_field(ch, "psi") for ch in range(len(sizes))])
    for other in got[1:]:
        for a, b in zip(got[0], other):
            assert np.array_equal(a, b)
