"""The row collide-stream kernel against the general one (EKPNP_LBM_ROWS=0),
each in its own launch: at the widths that a small context alone would take
through the one-launch kernel, and on a large channel.  The kernels round the
flux products of the storage references and one sum of squares differently, in
FP64; a stored FP32 value may then differ by a unit in its last place."""
import numpy as np
import pytest

from test_gpu_lbm_fwd import start

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny", [(64, 37), (128, 20), (256, 40), (192, 30), (2048, 512)])
def test_row_kernel_agrees_with_the_general_kernel(nx, ny, monkeypatch):
    # noise, walls and a flow along x; a channel of 320 nodes beside it keeps the launches apart
    steps, runs = 12, []
    for env in ("1", "0"):
        monkeypatch.setenv("EKPNP_LBM_ROWS", env)
        s = start([(nx, ny), (320, 6)], "fp32")
        s.step(steps)  # a re-centring at step 8
        runs.append({sp: s.get_populations(0, sp) for sp in ("f", "h", "g")})
        s.close()
    for sp in runs[0]:
        a, b = runs[0][sp], runs[1][sp]
        # stored deviations are at most of the populations' size: a last place of 2^-24 of it, one
        # more such step after step
        bound = steps * 2.0 ** -24 * np.abs(b).max()
        d = np.abs(a - b)
        print(f"{nx}x{ny} {sp}: {np.count_nonzero(d)} of {d.size} differ, largest {d.max():.1e}, bound {bound:.1e}",
              flush=True)
        assert d.max() <= bound
