"""FP32 rounding of the entry-balanced kernels that default plans run: rows of
one 1 and small entries of half its last place, each of which a sum in single
precision loses when it is added alone.  Products are exact, sums are below 2,
and 2^-24 is the largest rounding error of one addition."""
import numpy as np
import pytest

from gpu_util import run

pytestmark = pytest.mark.gpu
U = 2.0 ** -24


def _rows(sp, n, length, stride, seed=6):
    """n rows of `length` entries, `stride` columns apart from a random first one; the 1 anywhere."""
    rng = np.random.default_rng(seed)
    m = max(n, stride * length)
    first = rng.integers(0, m - stride * (length - 1), n)
    col = first[:, None] + np.arange(length) * stride
    val = np.full((n, length), U, np.float32)
    val[np.arange(n), rng.integers(0, length, n)] = 1.0
    row = np.repeat(np.arange(n), length)
    A = sp.Coo.from_arrays(n, m, row.astype(np.uint32), col.ravel().astype(np.uint32), val.ravel())
    return A, 1.0 + (length - 1) * U


@pytest.mark.parametrize("kern", ["CSR-nnz", "COO-nnz", "RBDCSR"])
@pytest.mark.parametrize("n,length,stride", [(40000, 33, 1), (160000, 20, 1), (50000, 40, 1), (90001, 36, 997)])
def test_wide_rounding(sp, ctx, kern, n, length, stride):
    """Tiles of 16 entries per thread.  Additions that meet the 1: rounding a thread's sum (once),
    three levels over the threads of a row, the waves before, the row's own thread, the tile before,
    and a second stripe."""
    A, want = _rows(sp, n, length, stride)
    y, plan = run(sp, ctx, kern, A, np.ones(A.ncols, np.float32))
    assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
    assert np.abs(y.astype(np.float64) - want).max() <= 8 * U
