"""The network's kernels at the edges of their 16-row tiles and 32-deep
products: batches around multiples of 16 and 32 and of the bias sums' 256 rows,
the narrowest layers, against the FP64 reference with BF16 rounding emulated."""
import numpy as np
import pytest

import mlp_ref as R
from ekpnp import surrogate as S

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,hidden,layers,n_out", [(1, 32, 1, 32), (15, 32, 1, 32), (16, 32, 2, 64),
                                                       (17, 96, 1, 32), (31, 32, 1, 160), (33, 64, 2, 32),
                                                       (255, 32, 1, 32), (257, 32, 1, 96)])
def test_forward_and_gradients_at_tile_edges(batch, hidden, layers, n_out):
    # a larger batch first: rows past the batch must not leak into its sums
    m = S.MLP(n_in=5, n_hidden=hidden, n_layers=layers, n_out=n_out, max_batch=300, seed=batch)
    shp = R.shapes(5, hidden, layers, n_out)
    p = m.get_params().astype(np.float64)
    rng = np.random.default_rng(batch)
    m.loss_grad(rng.uniform(-1, 1, (300, 5)), rng.standard_normal((300, n_out)))
    x = rng.uniform(-1, 1, (batch, 5))
    t = rng.standard_normal((batch, n_out)) * 0.5
    y, _ = R.forward(p, x, shp, emulate=True)
    e = float(np.linalg.norm(m.forward(x) - y) / np.linalg.norm(y))
    loss, g = m.loss_grad(x, t)
    lr, gr = R.loss_grad(p, x, t, shp, emulate=True)
    # FP32 sums of at most 300 terms in another order (relative 300 eps =
    # 2e-5 at worst), and a BF16 rounding that falls the other way here and there
    eg = float(np.linalg.norm(g - gr) / np.linalg.norm(gr))
    print("mlp tiles", batch, hidden, layers, n_out, e, eg, flush=True)
    assert e < 1e-4 and eg < 1e-4
    assert abs(loss - lr) <= 1e-5 * lr


def test_transposed_shadow_follows_training_and_set_params():
    # the backward pass reads the transposed weights: after training steps and
    # after set_params its gradients must be those of the current parameters
    m = S.MLP(n_in=5, n_hidden=64, n_layers=2, n_out=96, max_batch=40, seed=1)
    shp = R.shapes(5, 64, 2, 96)
    rng = np.random.default_rng(0)
    x, t = rng.uniform(-1, 1, (40, 5)), rng.standard_normal((40, 96))
    start = m.get_params()
    for _ in range(5):
        m.train_step(x, t, 1e-2)
    for params in (None, start):
        if params is not None:
            m.set_params(params)
        _, g = m.loss_grad(x, t)
        _, gr = R.loss_grad(m.get_params().astype(np.float64), x, t, shp, emulate=True)
        assert float(np.linalg.norm(g - gr) / np.linalg.norm(gr)) < 1e-4
