"""The collide-stream kernels' cached population planes: how many of the 27 go
through the caches depends on the size of the whole context and must change
nothing.  One channel advanced alone against copies of it
in batches on either side of each limit."""
import numpy as np
import pytest

import ekpnp

pytestmark = pytest.mark.gpu

NAMES = ("f", "h", "g")


def advance(nx, ny, precision, copies, compute):
    s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, kappa_h=4.0)] * copies, precision=precision, compute_fp64=compute)
    rng = np.random.default_rng(nx * ny)
    one, zero = np.ones((ny, nx)), np.zeros((ny, nx))
    fields = (one + 1e-3 * rng.standard_normal((ny, nx)), zero, zero, 1 + 0.1 * rng.random((ny, nx)),
              1 + 0.1 * rng.random((ny, nx)), 1e-2 * rng.standard_normal((ny, nx)))
    last = copies - 1
    for ch in {0, copies // 2, last}:
        s.set_fields(ch, *fields)
    s.init_equilibrium()
    for _ in range(3):
        s.stream_collide_save()
    lbm = [[s.get_populations(ch, n) for n in NAMES] for ch in (0, copies // 2, last)]
    s.step(3)
    full = [[s.get_populations(ch, n) for n in NAMES] for ch in (0, copies // 2, last)]
    s.close()
    return lbm, full


# both lattices of one copy: 13.8-14.2 MB (FP32 storage), 28.3 MB (FP64);
# row kernel: none below 80 MB, then 27, 18, 13, 9, 6, 4, 2 and no planes;
# k_lbm with FP32 storage: 27 up to 230 MB, then 13, 6, 2, or with
# narrow channels none; with FP64 storage: none,
# 27, 13, 9, 4
@pytest.mark.parametrize("nx,ny,precision,compute,batches", [
    (1024, 64, "fp32", True, (5, 6, 11, 12, 16, 20, 30, 45, 70, 100, 160)),
    (1000, 64, "fp32", True, (16, 17, 24, 45, 90)),
    (32, 256, "fp32", True, (130, 131)),
    (1000, 64, "fp32", False, (16, 17)),
    (1024, 64, "fp64", True, (2, 3, 8, 9, 12, 35)),
])
def test_cached_planes_change_nothing(nx, ny, precision, compute, batches):
    (want,), (want_full,) = [x[:1] for x in advance(nx, ny, precision, 1, compute)]
    for copies in batches:
        lbm, full = advance(nx, ny, precision, copies, compute)
        for got in lbm:  # collide-stream alone: the same bits
            for a, b in zip(got, want):
                assert np.array_equal(a, b), (copies, np.abs(a - b).max())
        # coupled: a batch may take another x-FFT kernel, whose psi differs in
        # the last bits; stored values then differ by an ulp of their storage
        # type (6e-8 of FP32), at most doubled by each of the steps' collisions
        for got in full:
            for a, b in zip(got, want_full):
                assert np.abs(a - b).max() <= 1e-6 * np.abs(b).max(), copies
