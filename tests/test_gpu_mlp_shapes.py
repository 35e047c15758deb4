"""The selector network's kernels at the edges of their tiles, against the
FP64 oracle: sizes around the 16-wide tiles, the largest networks one CU
holds and the first ones past them (which run layer by layer), sample counts
around a 16-sample tile and around one tile per workgroup.  Tolerances as for
the network's other gradient test: loss 1e-5, gradients 1e-4 of the largest.
The two ways to run a network give the same bits."""
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


@pytest.mark.parametrize("d,c,n", [(24, 22, 1920), (7, 3, 127), (24, 64, 129), (24, 12, 1)])
def test_one_cu_and_layers_give_the_same_bits(ctx, d, c, n):
    # 128 hidden units fit one CU, 129 run layer by layer; the last unit of
    # those has no weights, so it stays zero and adds zeros to every sum
    h = 128
    rng = np.random.default_rng(d * 100 + n)
    small, large = S.Mlp(ctx, d, h, c, seed=3), S.Mlp(ctx, d, h + 1, c, seed=3)

    def split(p, units):
        sizes = [d * units, units, units * units, units, units * c, c]
        at = np.cumsum([0] + sizes)
        shapes = [(d, units), (units,), (units, units), (units,), (units, c), (c,)]
        return [p[at[i]:at[i + 1]].reshape(shapes[i]) for i in range(6)]

    def without_last(p):
        w1, b1, w2, b2, w3, b3 = split(p, h + 1)
        return np.concatenate([w1[:, :h].ravel(), b1[:h], w2[:h, :h].ravel(), b2[:h], w3[:h].ravel(), b3])

    w1, b1, w2, b2, w3, b3 = split(small.get_params(), h)
    large.set_params(np.concatenate([np.pad(w1, ((0, 0), (0, 1))).ravel(), np.pad(b1, (0, 1)),
                                     np.pad(w2, (0, 1)).ravel(), np.pad(b2, (0, 1)),
                                     np.pad(w3, ((0, 1), (0, 0))).ravel(), b3]))
    small.set_params(small.get_params())
    x = rng.normal(0, 1, (n, d)).astype(np.float32)
    y = rng.integers(0, c, n).astype(np.int32)
    (l1, g1), (l2, g2) = small.loss_grad(x, y), large.loss_grad(x, y)
    assert l1 == l2 and np.array_equal(g1, without_last(g2))
    assert small.train(x, y, steps=6) == large.train(x, y, steps=6)
    assert np.array_equal(small.get_params(), without_last(large.get_params()))
    assert np.array_equal(small.predict(x)[0], large.predict(x)[0])
    small.free()
    large.free()
