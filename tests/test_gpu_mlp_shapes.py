"""The selector network's kernels at the edges of their tiles, against the
FP64 oracle: sizes around the 16-wide tiles, the largest networks one CU
holds and the first ones past them (which run layer by layer), sample counts
around a 16-sample tile and around one tile per workgroup.  Tolerances as for
the network's other gradient test: loss 1e-5, gradients 1e-4 of the largest."""
import numpy as np
import pytest

from clspmv_amd import selector as S
from oracle import mlp_oracle as MO

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d,h,c,n", [
    (1, 1, 2, 1), (16, 16, 16, 16), (17, 17, 17, 17), (15, 31, 33, 15), (24, 128, 22, 1920), (24, 128, 48, 100),
    (64, 96, 22, 33), (24, 128, 64, 50), (65, 40, 5, 40), (20, 129, 9, 70), (8, 20, 65, 60),
    (24, 64, 22, 4096), (24, 64, 22, 4097), (10, 112, 12, 9001),
])
def test_loss_gradients_and_logits(ctx, d, h, c, n):
    rng = np.random.default_rng(d * 7919 + h * 101 + c + n)
    net = S.Mlp(ctx, d, h, c, seed=5)
    p = net.get_params()
    x = rng.normal(0, 1, (n, d)).astype(np.float32)
    y = rng.integers(0, c, n).astype(np.int32)
    loss, g = net.loss_grad(x, y)
    loss64, g64 = MO.loss_grad(p, x, y, d, h, c)
    assert abs(loss - loss64) <= 1e-5 * max(1.0, abs(loss64))
    scale = np.max(np.abs(g64))
    assert np.max(np.abs(g - g64)) <= 1e-4 * scale, np.max(np.abs(g - g64)) / scale
    z, _ = net.predict(x)
    z64 = MO.forward(p, x, d, h, c)[2]
    assert np.max(np.abs(z - z64)) <= 1e-4 * np.max(np.abs(z64))
    net.free()
