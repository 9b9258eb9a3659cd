"""BCSR 4 x 4 blocks times 8, 16 and mixed column counts (matrix cores for FP32
and FP64): block rows of 0 to 130 blocks around the step and batch sizes, a
last block column and row that are cut, and x pieces that are not aligned."""
import numpy as np
import pytest

from gpu_util import assert_parity_multi

pytestmark = pytest.mark.gpu
COUNTS = [0, 1, 3, 15, 16, 17, 31, 32, 33, 63, 64, 65, 127, 128, 130, 2]


@pytest.mark.parametrize("k,ldx", [(8, 8), (8, 9), (16, 16), (16, 18), (27, 28)])
@pytest.mark.parametrize("cut", [0, 3])
@pytest.mark.parametrize("dt", [4, 5])
def test_block_rows(sp, ctx, dt, cut, k, ldx):
    rng = np.random.default_rng(7)
    n, m = 4 * len(COUNTS) * 3 - cut, 4 * 140 - cut
    row, col = [], []
    for I, c in enumerate(COUNTS * 3):
        for J in np.sort(rng.choice(140, c, replace=False)):
            i, j = np.meshgrid(np.arange(4), np.arange(4), indexing="ij")
            keep = rng.random((4, 4)) < 0.7
            keep[0, 0] = True
            row.append((4 * I + i)[keep])
            col.append((4 * J + j)[keep])
    row, col = np.concatenate(row), np.concatenate(col)
    ok = (row < n) & (col < m)
    row, col = row[ok], col[ok]
    o = np.lexsort((col, row))
    t = sp.NP_DTYPE[dt]
    A = sp.Coo.from_arrays(n, m, row[o].astype(np.uint32), col[o].astype(np.uint32), rng.uniform(-1, 1, len(o)).astype(t))
    X = rng.uniform(-1, 1, (m, ldx)).astype(t)
    for kern in ("BCSR-block", "BCSR-nnz", "BCOO-nnz"):
        plan = sp.Plan(ctx, kern, A)
        xd = sp.DeviceArray.from_numpy(ctx, X)
        yd = sp.DeviceArray(ctx, (n, ldx), t)
        yd.fill_bytes(0x5A)
        plan.spmm(k, xd.addr, ldx, yd.addr, ldx)
        ctx.sync()
        Y = yd.numpy()
        assert_parity_multi(dt, np.ascontiguousarray(Y[:, :k]), A, np.ascontiguousarray(X[:, :k]), f"{kern} k{k}")
        assert np.all(np.ascontiguousarray(Y[:, k:]).view(np.uint8) == 0x5A)
