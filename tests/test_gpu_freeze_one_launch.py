"""A channel that run_to_residual freezes inside a small context, whose
collide-stream launch holds the transforms of both steps (two spectra in
use, the frozen state in either lattice): the frozen channel and the ones that
run on have the bits of the same run on separate launches, which one wide channel
more brings about."""
import numpy as np
import pytest

import ekpnp
from test_gpu_lbm_fwd import same, state

pytestmark = pytest.mark.gpu


# the row kernel, k_lbm, both; from an odd step on, the frozen state sits in the
# other lattice half of the time
@pytest.mark.parametrize("precision", ["fp32", "fp64"])
@pytest.mark.parametrize("every", [20, 64])
@pytest.mark.parametrize("sizes", [[(64, 12), (128, 40), (64, 16)], [(32, 12), (10, 40), (4, 20)],
                                   [(64, 12), (32, 40), (20, 16)]])
def test_frozen_channel(sizes, every, precision):
    def run(more):
        s = ekpnp.Solver([ekpnp.lattice_params(nx, ny, tau=1.0, zeta=-0.5, kappa_h=1.5, e_x=1e-4)
                          for nx, ny in sizes + more], precision=precision)
        s.initialization(ekpnp.COLD_NOISE, 9)
        s.init_equilibrium()
        s.step(1)
        steps = s.run_to_residual(1e-7, every, 200000)
        out = [state(s, ch) for ch in range(len(sizes))]
        s.step(5)  # all channels move on again
        out += [state(s, ch) for ch in range(len(sizes))]
        s.close()
        return steps[:len(sizes)], out

    (na, a), (nb, b) = run([]), run([(320, 14)])
    print(sizes, every, precision, na, flush=True)
    assert np.array_equal(na, nb)
    assert na.min() > 0 and len(set(na.tolist())) > 1  # some were frozen while others ran
    for k, (x, y) in enumerate(zip(a, b)):
        if k < len(sizes) or nb.max() == na.max():
            same(x, y, (sizes[k % len(sizes)], every))
