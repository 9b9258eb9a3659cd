"""Batches that mix plans of every kind (wide tiles of skewed and even rows,
panels, row kernels, blocks), element types of 8 bytes and column counts, over
several replays with new inputs."""
import numpy as np
import pytest

from gpu_util import assert_parity_multi

pytestmark = pytest.mark.gpu
COUNTS = [1, 2, 8, 32, 43]


@pytest.mark.parametrize("turn", range(5))
@pytest.mark.parametrize("dt", [3, 5])
def test_mixed_plans(sp, ctx, dt, turn):
    mats = [("CSR-nnz", sp.gen_rmat(13, 100000, dtype=dt, seed=1)), ("CSR-nnz", sp.gen_banded(40000, 64, 2, 64, dtype=dt, seed=2)),
            ("COO-nnz", sp.gen_rmat(12, 50000, dtype=dt, seed=3)), ("BCOO-nnz", sp.gen_stencil27(9, 4, True, dt, seed=4)),
            ("CSR-row", sp.gen_uniform(3001, 3001, 2, 64, dtype=dt, seed=5)), ("BCSR-block", sp.gen_stencil27(8, 4, True, dt, seed=6))]
    plans = [sp.Plan(ctx, kern, A) for kern, A in mats]
    ks = [COUNTS[(i + turn) % 5] for i in range(len(mats))]
    batch = sp.Batch(ctx, plans, ks)
    X = [None] * len(mats)
    yd = [sp.DeviceArray(ctx, (A.nrows, k), sp.NP_DTYPE[dt]) for (_, A), k in zip(mats, ks)]
    xd = [sp.DeviceArray(ctx, (A.ncols, k), sp.NP_DTYPE[dt]) for (_, A), k in zip(mats, ks)]
    for rep in range(3):
        for i, ((_, A), k) in enumerate(zip(mats, ks)):
            X[i] = np.stack([sp.gen_vector(dt, A.ncols, seed=50 * rep + 9 * i + q) for q in range(k)], axis=1)
            xd[i].upload(X[i])
            yd[i].fill_bytes(0x5A)
        batch.run([x.addr for x in xd], [y.addr for y in yd])
        ctx.sync()
        for i, (kern, A) in enumerate(mats):
            assert_parity_multi(dt, yd[i].numpy(), A, X[i], f"{kern} k{ks[i]} replay {rep}")
