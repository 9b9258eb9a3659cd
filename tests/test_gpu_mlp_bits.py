"""The two-kernel loss and gradient of the selector MLP against its layer
kernels, bit for bit: a network with one input more, whose weights and values
are zero, takes the layer kernels (its width is no multiple of 8) and has the
same sums."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,B", [((64, 128, 128, 25), b) for b in (1, 16, 63, 64, 65, 257)] +
                         [((8, 8, 16, 1), 5), ((248, 256, 256, 256), 67), ((72, 136, 200, 129), 66)])
def test_same_bits(sp, ctx, sizes, B):
    i, h1 = sizes[:2]
    r = np.random.default_rng(B)
    X = r.normal(0, 1, (B, i)).astype(np.float32)
    T = r.normal(0, 1, (B, sizes[-1])).astype(np.float32)
    M = (r.random((B, sizes[-1])) < 0.9).astype(np.float32)
    two, layers = sp.Mlp(ctx, sizes, seed=3), sp.Mlp(ctx, (i + 1,) + sizes[1:], seed=3)
    p = two.get_params()
    wide = np.zeros((h1, i + 1), p.dtype)
    wide[:, :i] = p[: h1 * i].reshape(h1, i)
    layers.set_params(np.concatenate([wide.ravel(), p[h1 * i:]]))
    X1 = np.concatenate([X, np.zeros((B, 1), np.float32)], axis=1)
    for mask in (M, None):
        L, g = two.loss_grad(X, T, mask)
        L1, g1 = layers.loss_grad(X1, T, mask)
        w = g1[: h1 * (i + 1)].reshape(h1, i + 1)
        assert L == L1 and not w[:, i].any()
        assert np.array_equal(g, np.concatenate([w[:, :i].ravel(), g1[h1 * (i + 1):]]))
