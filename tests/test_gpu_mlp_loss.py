"""The network's loss is the mean of the squared errors to the last bit of the
float it is returned in, also where a few large errors stand beside small ones."""
import math

import numpy as np
import pytest

from ekpnp import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,n_out", [(16, 64), (64, 64), (33, 96)])
def test_small_errors_beside_a_large_one_count(batch, n_out):
    m = S.MLP(n_in=5, n_hidden=32, n_layers=1, n_out=n_out, max_batch=64)
    m.set_params(np.zeros_like(m.get_params()))  # outputs are exactly 0: the errors are the targets
    # 2^24 and terms below half its spacing in FP32, which a running FP32 sum drops one by one
    t = np.zeros((batch, n_out), dtype=np.float32)
    t[::16, ::16] = 4096.0
    for r in range(1, 4):
        t[r::16, ::16] = 0.995
    t[::16, 1::16] = t[::16, 2::16] = t[::16, 4::16] = t[::16, 8::16] = 0.995
    loss, _ = m.loss_grad(np.ones((batch, 5)), t)
    want = math.fsum(float(v) ** 2 for v in t.ravel()) / t.size
    # one rounding of an FP64 sum: half a unit in the last place (and the FP64 sum's own error)
    assert abs(loss - want) <= 0.501 * np.spacing(np.float32(want))
