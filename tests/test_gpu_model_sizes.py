"""GPU test of the cost model's gradient at the edges of its tiles: one sample,
a whole tile of 64, one more, and one more partial gradient than the sum takes
at a time (16), against the numpy statement."""
import sys

import mlp_ref
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def say(*a):
    print("[gpu-case]", *a, file=sys.stderr, flush=True)


@pytest.mark.parametrize("m", [1, 64, 65, 1024, 1025])
def test_gradient_at_tile_edges(bh, m):
    say("model sizes", m)
    rng = np.random.default_rng(m)
    p = mlp_ref.init(5)
    x = rng.normal(size=(m, 8)).astype(np.float32)
    x[::3, 6] = x[::3, 5]          # closed gates
    t = (0.2 * rng.normal(size=m)).astype(np.float32)
    with bh.Engine() as eng:
        eng.model_set_params(p)
        g, loss = eng.model_gradients(x, t)
    lr, gr = mlp_ref.loss_and_grad(p, x, t, dtype=np.float64)
    # FP32 sums of at most 1025 terms: 1025 x 2^-24 of the largest entry's scale
    assert abs(loss - lr) <= 1e-4 * max(lr, 1e-6)
    assert np.abs(g - gr).max() <= 1e-4 * max(np.abs(gr).max(), 1e-6)
