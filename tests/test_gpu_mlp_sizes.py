"""The predictor's gradient, training and scale kernels at the row counts
where they can go wrong (one row, a sample block and one more or less, a
reduction of 64 partials and one more, the scale's 16 rows per thread),
against FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from heddlemd_amd.engine import ShakePredictor  # noqa: E402
from tests.test_gpu_shake_mlp import _rows  # noqa: E402


@pytest.mark.parametrize("n", [1, 63, 64, 65, 4096, 4097, 16384, 16385, 40001])
def test_gradient_and_scale_at_edge_sizes(oracle, n):
    print(f"case: {n} rows", flush=True)
    rng = np.random.default_rng(n)
    x, t = _rows(rng, n, 3e-3)
    m = ShakePredictor(seed=5)
    # the first training call fixes the scale: the rms of column 0
    m.train(x, t, epochs=1, batch=4096, lr=1e-4)
    p = m.params
    scale = np.sqrt(np.mean(x[:, 0].astype(np.float64) ** 2))
    assert p[-1] == pytest.approx(scale, rel=2e-7)  # one f32 rounding
    loss, g = m.gradient(x, t)
    lref, gref = oracle.mlp_loss_grad(p.astype(np.float64), x, t)
    # f32 sums of up to 64 terms per block and n / 64 blocks, device tanhf
    assert np.linalg.norm(g - gref) <= 1e-4 * np.linalg.norm(gref)
    assert loss == pytest.approx(lref, rel=1e-4)
    m.close()
