"""Infinities and NaN in x, in some right-hand sides only, and in the matrix:
a row that meets one has the class of its exact sum, and no other row and no
other column of the result changes.  Blocks multiply their padding, so all rows
of a block that holds such a column may be non-finite."""
import numpy as np
import pytest

from gpu_util import assert_parity_multi, run

pytestmark = pytest.mark.gpu


def _matrix(sp, dt, name):
    rng = np.random.default_rng(12)
    if name == "hub":  # skewed: one row over many tiles
        n, m = 5000, 70001
        row = np.concatenate([np.full(52000, 17), rng.integers(0, n, 30000)])
        col = rng.integers(0, m, row.size)
    elif name == "even":  # 2 to 64 entries in a row near the diagonal, 1.3M together
        n = m = 40000
        row = np.repeat(np.arange(n), rng.integers(2, 65, n))
        col = (row + rng.integers(0, 64, row.size)) % m
    else:  # 4 x 4 blocks, cut at the last row and column
        n, m = 4 * 900 - 2, 4 * 800 - 3
        I = np.repeat(np.arange(900), rng.integers(0, 60, 900))
        J = rng.integers(0, 800, I.size)
        i, j, _ = np.meshgrid(np.arange(4), np.arange(4), I, indexing="ij")
        row, col = (4 * I + i).ravel(), (4 * J + j).ravel()
        keep = (row < n) & (col < m) & (rng.random(row.size) < 0.7)
        row, col = row[keep], col[keep]
    key = np.unique(row.astype(np.uint64) * np.uint64(m) + col.astype(np.uint64))
    t = sp.NP_DTYPE[dt]
    return sp.Coo.from_arrays(n, m, (key // m).astype(np.uint32), (key % m).astype(np.uint32),
                              rng.uniform(0.5, 1, key.size).astype(t) * rng.choice([-1, 1], key.size).astype(t))


def _check(dt, Y, A, X, block, what):
    """Y against the finite parts' oracle where a row meets only finite numbers, else by class."""
    for q in range(X.shape[1]):
        with np.errstate(invalid="ignore"):
            terms = A.values.astype(np.float64) * X[A.colind, q].astype(np.float64)
        bad = ~np.isfinite(terms)
        nan, pos, neg = (np.bincount(A.rowind[bad], w[bad], A.nrows) > 0 for w in
                         (np.isnan(terms).astype(float), (terms == np.inf).astype(float), (terms == -np.inf).astype(float)))
        hit = nan | pos | neg
        y = Y[:, q].astype(np.float64)
        if block > 1:  # a padded entry of a bad column in one of the block's rows
            touched = np.isin(A.colind // block, np.unique(np.nonzero(~np.isfinite(X[:, q]))[0] // block))
            rows = np.unique(A.rowind[touched] // block)
            clean = ~np.isin(np.arange(A.nrows) // block, rows) & ~hit
            assert not np.isfinite(y[hit]).any(), (what, q)
        else:
            clean = ~hit
            assert np.isnan(y[nan | (pos & neg)]).all(), (what, q)
            assert (y[pos & ~neg & ~nan] == np.inf).all() and (y[neg & ~pos & ~nan] == -np.inf).all(), (what, q)
        assert np.isfinite(y[clean]).all(), (what, q, np.nonzero(clean & ~np.isfinite(y))[0][:5])
        if q in (0, X.shape[1] - 1):
            yes = clean[A.rowind] & ~bad
            F = type(A).from_arrays(A.nrows, A.ncols, A.rowind[yes], A.colind[yes], A.values[yes])
            xf = np.where(np.isfinite(X[:, q]), X[:, q], 0).astype(X.dtype)
            yf = np.where(clean, Y[:, q], 0).astype(X.dtype)
            assert_parity_multi(dt, yf[:, None], F, xf[:, None], f"{what} rhs {q}")


@pytest.mark.parametrize("kern,name,k", [
    ("CSR-nnz", "hub", 1), ("COO-nnz", "hub", 1), ("CSR-nnz", "even", 1), ("RBDCSR", "even", 1),
    ("CSR-nnz", "hub", 8), ("COO-nnz", "hub", 35), ("CSR-nnz", "even", 2), ("CSR-nnz", "even", 16),
    ("BCSR-nnz", "blocks", 1), ("BCSR-nnz", "blocks", 8), ("BCSR-block", "blocks", 16), ("BCOO-nnz", "blocks", 1),
    ("BCOO-nnz", "blocks", 8), ("BCOO-block", "blocks", 16)])
@pytest.mark.parametrize("dt", [4, 5])
def test_rows_keep_to_themselves(sp, ctx, dt, kern, name, k):
    A = _matrix(sp, dt, name)
    block = 4 if name == "blocks" else 1
    rng = np.random.default_rng(k)
    X = rng.uniform(0.5, 1, (A.ncols, k)).astype(sp.NP_DTYPE[dt])
    plan = sp.Plan(ctx, kern, A)
    bad = [(0, np.nan), (A.ncols - 1, np.inf), (A.ncols // 2, -np.inf)]
    for some in (bad, bad[1:2], []):
        Z = X.copy()
        for c, v in some:
            Z[c, ::2] = v  # every second right-hand side stays finite
        Y, _ = run(sp, ctx, kern, A, Z[:, 0] if k == 1 else Z, k=k, plan=plan)
        _check(dt, Y.reshape(A.nrows, k), A, Z, block, f"{kern} k{k} {len(some)}")
    V = A.values.copy()
    at = rng.choice(V.size, 3, replace=False)
    V[at] = [np.nan, np.inf, -np.inf]
    B = sp.Coo.from_arrays(A.nrows, A.ncols, A.rowind, A.colind, V)
    Y, _ = run(sp, ctx, kern, B, X[:, 0] if k == 1 else X, k=k)
    _check(dt, Y.reshape(A.nrows, k), B, X, block, f"{kern} k{k} values")


@pytest.mark.parametrize("k", [1, 8])
@pytest.mark.parametrize("dt", [4, 5])
def test_overflow(sp, ctx, dt, k):
    """Rows whose sum is beyond the largest number are infinite, the rows around them exact."""
    t = sp.NP_DTYPE[dt]
    big = np.finfo(t).max
    n, per = 40000, 33
    row = np.repeat(np.arange(n), per)
    col = (row + np.tile(np.arange(per), n)) % n
    key = np.sort(row.astype(np.uint64) * np.uint64(n) + col.astype(np.uint64))
    row, col = (key // n).astype(np.uint32), (key % n).astype(np.uint32)
    val = np.ones(row.size, t)
    val[row % 100 == 7] = big
    val[row % 100 == 8] = -big
    hub = np.arange(n, dtype=np.uint32)  # skewed, so that the entry-balanced kernels run
    A = sp.Coo.from_arrays(n + 1, n, np.concatenate([row, np.full(n, n, np.uint32)]), np.concatenate([col, hub]),
                           np.concatenate([val, np.ones(n, t)]))
    Y, plan = run(sp, ctx, "CSR-nnz", A, np.ones(n if k == 1 else (n, k), t), k=k)
    assert k > 1 or plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
    r = np.arange(n + 1) % 100
    want = np.where(r == 7, np.inf, np.where(r == 8, -np.inf, per)).astype(t)
    want[n] = n
    assert (Y.reshape(n + 1, k) == want[:, None]).all()
