"""The network on batches of more row tiles than one dimension of a launch
holds (65536 of 16 rows), and on the warm-start network's own layers above its
training batch."""
import numpy as np
import pytest

import mlp_ref as R
from ekpnp import surrogate as S

pytestmark = pytest.mark.gpu


# 65535 row tiles (one launch), 65538 and 67584 (two)
@pytest.mark.parametrize("batch", [1048560, 1048600, 1081344])
def test_more_row_tiles_than_a_launch_dimension(batch):
    net = S.MLP(n_in=5, n_hidden=32, n_layers=1, n_out=32, max_batch=batch, seed=3)
    ref = S.MLP(n_in=5, n_hidden=32, n_layers=1, n_out=32, max_batch=4096, seed=3)
    rng = np.random.default_rng(1)
    x = rng.uniform(-1, 1, (batch, 5)).astype(np.float32)
    y = net.forward(x)
    half = (batch + 31) // 32 * 16
    for a in (0, half - 2048, 1048560 - 4096, batch - 4096):  # a row's outputs depend on that row alone
        assert np.array_equal(y[a:a + 4096], ref.forward(x[a:a + 4096])), a
    # targets that the network meets exactly but for 264 rows, before (beyond one launch's: on
    # both sides of) its last row and at the end
    edge = min(1048560, batch - 198)
    rows = np.r_[edge - 66:edge + 66, batch - 132:batch]
    t = y.copy()
    t[rows] += rng.standard_normal((264, 32)).astype(np.float32)
    loss, g = net.loss_grad(x, t)
    want = float(np.sum((y[rows] - t[rows]).astype(np.float64) ** 2)) / t.size
    assert abs(loss - want) <= 1.2e-7 * want  # rounded to FP32 once
    if batch % 264 == 0:  # 4096 x 264: the gradient of those rows alone, scaled by a power of two
        _, gr = ref.loss_grad(x[rows], t[rows])
        # both sum 264 terms in FP32, grouped by their places in the batch
        assert np.linalg.norm(g * np.float32(batch // 264) - gr) <= 264 * 2.0 ** -24 * np.linalg.norm(gr) * 4


@pytest.mark.parametrize("batch", [511, 1000])
def test_warm_start_network_above_its_training_batch(batch):
    m = S.MLP(max_batch=batch, seed=batch)
    shp = R.shapes(S.N_IN, 256, 4, S.N_OUT)
    p = m.get_params().astype(np.float64)
    rng = np.random.default_rng(batch)
    x, t = rng.uniform(-1, 1, (batch, S.N_IN)), 0.5 * rng.standard_normal((batch, S.N_OUT))
    y, _ = R.forward(p, x, shp, emulate=True)
    loss, g = m.loss_grad(x, t)
    lr, gr = R.loss_grad(p, x, t, shp, emulate=True)
    e = float(np.linalg.norm(m.forward(x) - y) / np.linalg.norm(y))
    eg = float(np.linalg.norm(g - gr) / np.linalg.norm(gr))
    print("warm-start network", batch, e, eg, flush=True)
    # BF16 roundings that fall the other way after an FP32 sum in another order: at most a few in
    # a thousand of 2^-9 each through four layers
    assert e < 1e-3 and eg < 1e-3
    assert abs(loss - lr) <= 1e-4 * lr
