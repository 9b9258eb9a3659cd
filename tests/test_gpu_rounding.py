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
@pytest.mark.parametrize("n,length,stride", [(112000, 33, 1), (190000, 20, 1), (92000, 40, 1), (90001, 36, 997)])
def test_wide_rounding(sp, ctx, kern, n, length, stride):
    """Tiles of 16 entries per thread.  Additions that meet the 1: rounding a thread's sum (once),
    three levels over the threads of a row, the waves before, the row's own thread, the tile before,
    and a second stripe."""
    A, want = _rows(sp, n, length, stride)
    y, plan = run(sp, ctx, kern, A, np.ones(A.ncols, np.float32))
    assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
    assert np.abs(y.astype(np.float64) - want).max() <= 8 * U


@pytest.mark.parametrize("k", [2, 8, 32])
@pytest.mark.parametrize("skewed", [True, False])
def test_panel_rounding(sp, ctx, k, skewed):
    """Groups of 16 entries.  Additions that meet the 1: rounding a group's sum (once), five levels
    over the groups of a wave, three waves before, the row's own group, the workgroups before."""
    A, want = _rows(sp, 9001, 33, 1)
    if skewed:  # a row of many entries, each of value 0
        extra = np.arange(A.ncols, dtype=np.uint32)
        A = sp.Coo.from_arrays(A.nrows + 1, A.ncols, np.concatenate([A.rowind, np.full(A.ncols, A.nrows, np.uint32)]),
                               np.concatenate([A.colind, extra]), np.concatenate([A.values, np.zeros(A.ncols, np.float32)]))
    Y, _ = run(sp, ctx, "CSR-nnz", A, np.ones((A.ncols, k), np.float32), k=k)
    err = np.abs(Y[:9001].astype(np.float64) - want)
    assert err.max() <= 11 * U and not Y[9001:].any()


@pytest.mark.parametrize("kern,k", [("CSR-nnz", 1), ("COO-row", 1), ("CSR-row", 8), ("CSR-row", 16)])
def test_fp64_rounding(sp, ctx, kern, k):
    """Rows of nine entries in threads or groups of eight: additions that meet the 1 are the rounding
    of its thread's sum, the other thread's and the tile's before."""
    n, u = 180000, 2.0 ** -53
    rng = np.random.default_rng(9)
    col = np.arange(n)[:, None] + np.arange(9)
    val = np.full((n, 9), u)
    val[np.arange(n), rng.integers(0, 9, n)] = 1.0
    A = sp.Coo.from_arrays(n, n + 8, np.repeat(np.arange(n, dtype=np.uint32), 9), col.ravel().astype(np.uint32), val.ravel())
    Y, _ = run(sp, ctx, kern, A, np.ones((n + 8, k) if k > 1 else n + 8), k=k)
    assert np.abs((Y - 1.0) - 8 * u).max() <= 3 * u


@pytest.mark.parametrize("dt", [4, 5])
@pytest.mark.parametrize("rc,ks", [((4, 4), (1, 8, 16, 32, 43)), ((2, 2), (1, 16)), ((2, 4), (1, 16, 32)),
                                   ((4, 2), (1, 32)), ((8, 8), (1, 2, 16))])
def test_bcoo_rounding(sp, ctx, dt, rc, ks):
    """Default BCOO plans, whatever kernel serves a width, are as accurate as the block-balanced kernel
    (algo=2): root mean square errors of 23000 sums or more, known to about 0.5%, within 2%."""
    A = sp.gen_stencil27(18, 4, True, dt, seed=3)
    rng = np.random.default_rng(4)
    t = sp.NP_DTYPE[dt]
    val = rng.uniform(-1, 1, A.nnz).astype(t)
    row, col = A.rowind.copy(), A.colind.copy()
    A = sp.Coo.from_arrays(A.nrows, A.ncols, row, col, val)
    starts = np.flatnonzero(np.r_[True, row[1:] != row[:-1]])
    o = {"row_block_size": rc[0], "col_block_size": rc[1]}
    plan, balanced = sp.Plan(ctx, "BCOO-nnz", A, sp.opts(**o)), sp.Plan(ctx, "BCOO-nnz", A, sp.opts(algo=2, **o))
    for k in ks:
        X = rng.uniform(-1, 1, (A.ncols, k) if k > 1 else A.ncols).astype(t)
        Y = [run(sp, ctx, "BCOO-nnz", A, X, k=k, plan=p)[0].reshape(A.nrows, k) for p in (plan, balanced)]
        X = X.reshape(A.ncols, k)
        err = np.zeros(2)
        for q in {0, 1, k // 2, k - 1} & set(range(k)):
            want = np.add.reduceat(val.astype(np.longdouble) * X[col, q].astype(np.longdouble), starts)
            err += [float(((y[:, q] - want) ** 2).mean()) for y in Y]
        assert err[0] <= 1.02 ** 2 * err[1], (k, np.sqrt(err))
