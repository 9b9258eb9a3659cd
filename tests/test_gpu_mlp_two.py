"""Loss and gradient of the selector MLP in two kernels against the CPU oracle:
batches around the tile edges, the narrowest and widest layers the path takes,
widths it leaves to the layer kernels, and no mask."""
import os
import sys

import numpy as np
import pytest

sys.path.insert(0, os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "oracle"))
import mlp_oracle as mo  # noqa: E402

pytestmark = pytest.mark.gpu
SIZES = (64, 128, 128, 25)


@pytest.mark.parametrize("sizes,B", [(SIZES, b) for b in (1, 2, 63, 64, 65, 257, 512)] +
                         [((8, 8, 16, 1), 5), ((256, 256, 256, 256), 67), ((72, 136, 200, 129), 66),
                          ((10, 20, 12, 3), 33), ((64, 264, 128, 25), 40)])
def test_loss_grad(sp, ctx, sizes, B):
    r = np.random.default_rng(B)
    X = r.normal(0, 1, (B, sizes[0])).astype(np.float32)
    T = r.normal(0, 1, (B, sizes[-1])).astype(np.float32)
    M = (r.random((B, sizes[-1])) < 0.9).astype(np.float32)
    m = sp.Mlp(ctx, sizes, seed=3)
    shapes, offs, n = mo.layout(sizes)
    bounds = offs + [n]
    for mask in (M, None):
        L, g = m.loss_grad(X, T, mask)
        Lw, gw = mo.loss_grad(m.get_params(), sizes, X, T, np.ones_like(T) if mask is None else mask)
        assert abs(L - Lw) <= 1e-5 * abs(Lw)
        for j in range(6):
            a, b = bounds[j], bounds[j + 1]
            assert np.abs(g[a:b] - gw[a:b]).max() <= 1e-4 * np.abs(gw[a:b]).max() + 1e-9, j
    g2 = m.loss_grad(X[: max(1, B // 2)], T[: max(1, B // 2)], None)[1]  # a smaller batch in the same buffers
    gw = mo.loss_grad(m.get_params(), sizes, X[: max(1, B // 2)], T[: max(1, B // 2)], np.ones_like(T[: max(1, B // 2)]))[1]
    assert np.abs(g2 - gw).max() <= 1e-4 * np.abs(gw).max() + 1e-9
