"""Wide column-ordered tiles and panels (automatic 1D CSR and COO plans): integers
bit-exact against the oracle, floats within the gamma(len+2) bound of the
long-double reference, at the edges of tiles, with rows crossing many tiles,
empty rows anywhere, columns further apart than a key holds, other leading
dimensions and batches."""
import numpy as np
import pytest

from gpu_util import assert_parity, assert_parity_multi, run

pytestmark = pytest.mark.gpu


def _coo(sp, dt, nrows, ncols, row, col, seed=3):
    key = np.unique(row.astype(np.uint64) * np.uint64(ncols) + col.astype(np.uint64))
    r, c = (key // ncols).astype(np.uint32), (key % ncols).astype(np.uint32)
    rng = np.random.default_rng(seed)
    t = sp.NP_DTYPE[dt]
    v = rng.integers(-4, 5, len(r)).astype(t) if dt <= 3 else rng.uniform(-1, 1, len(r)).astype(t)
    return sp.Coo.from_arrays(nrows, ncols, r, c, v)


def _x(sp, dt, shape, seed=5):
    rng = np.random.default_rng(seed)
    t = sp.NP_DTYPE[dt]
    return rng.integers(-4, 5, shape).astype(t) if dt <= 3 else rng.uniform(-1, 1, shape).astype(t)


def _pattern(name, rng):
    """(rows, columns, row index, column index): row lengths and columns of one matrix."""
    if name == "hub":  # one row over many tiles, then short ones: skewed
        n, m = 5000, 70001
        row = np.concatenate([np.full(52000, 17), rng.integers(0, n, 30000)])
        return n, m, row, rng.integers(0, m, row.size)
    if name == "empties":  # empty rows first, last and in long gaps
        n, m = 60000, 3001
        row = np.concatenate([rng.integers(500, 900, 20000), rng.integers(41000, 41300, 20000), np.full(2500, 700)])
        return n, m, row, rng.integers(0, m, row.size)
    if name == "far":  # columns beyond 32 bits less the tile's positions: runs end early at a row's wrap
        n, m = 300, (1 << 22) + 13
        row = np.repeat(np.arange(12), 9000)
        col = (np.tile(np.arange(9000), 12) * (m // 9000) + row).clip(max=m - 1)
        extra = rng.integers(0, n, 2000)
        return n, m, np.concatenate([row, extra]), np.concatenate([col, rng.integers(0, m, 2000)])
    if name == "one":  # a single row and one entry more
        n, m = 900, 65000
        return n, m, np.concatenate([np.full(60000, 3), [899]]), np.concatenate([np.arange(60000), [64999]])
    # exact: whole tiles of 4096, 8192 and 16384 entries, last row ending with the last tile
    n, m = 1024, 4096
    row = np.concatenate([np.repeat(np.arange(n), 28), np.full(4096, 1000)])
    return n, m, row, np.concatenate([np.tile(np.arange(28) * 3, n), np.arange(4096)])


@pytest.mark.parametrize("name", ["hub", "empties", "far", "one", "exact"])
@pytest.mark.parametrize("dt", [0, 1, 2, 3, 4, 5])
def test_wide_parity(sp, ctx, dt, name):
    n, m, row, col = _pattern(name, np.random.default_rng(11))
    A = _coo(sp, dt, n, m, row, col)
    x = _x(sp, dt, m)
    for kern in ("CSR-nnz", "CSR-row", "COO-nnz", "COO-row"):
        y, plan = run(sp, ctx, kern, A, x)
        assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
        assert_parity(dt, y, A, x, f"{kern}/{name}")


@pytest.mark.parametrize("dt,rows,per,band", [(4, 40000, 33, 64), (4, 330000, 5, 16), (5, 40000, 33, 64), (0, 70001, 48, 64),
                                              (4, 100003, 40, 100003), (5, 100003, 24, 100003), (2, 9001, 33, 9001)])
def test_wide_even_rows(sp, ctx, dt, rows, per, band):
    """The shapes of even rows: local and scattered columns, 4- and 8-byte sums, more than 3M entries."""
    rng = np.random.default_rng(rows)
    row = np.repeat(np.arange(rows), per)
    col = (row + rng.integers(0, band, row.size)) % rows
    A = _coo(sp, dt, rows, rows, row, col)
    x = _x(sp, dt, rows)
    for kern in ("CSR-nnz", "COO-nnz-rgrn"):
        y, plan = run(sp, ctx, kern, A, x)
        assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
        assert_parity(dt, y, A, x, kern)


@pytest.mark.parametrize("kern", ["RBDCSR", "BDCSR", "DCSR", "RBDCOO", "DCOO"])
@pytest.mark.parametrize("dt", [0, 4, 5])
def test_wide_tilings(sp, ctx, dt, kern):
    """2D tilings: long gaps of empty rows in every stripe, a stripe without entries, a wide panel."""
    rng = np.random.default_rng(4)
    n = 45011
    row = np.repeat(np.arange(n), 33)
    col = (row + rng.integers(0, 64, row.size)) % n
    A = _coo(sp, dt, n, n, row, col)
    B = _coo(sp, dt, n, 2 * n, row, col)  # the second of two stripes is empty
    for M in (A, B):
        x = _x(sp, dt, M.ncols)
        y, plan = run(sp, ctx, kern, M, x)
        if "COO" in kern or (M is A and kern != "DCSR"):  # (CSR: no empty tile)
            assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED
        assert_parity(dt, y, M, x, kern)
        y, _ = run(sp, ctx, kern, M, x, plan=plan)
        assert_parity(dt, y, M, x, kern)
    X = _x(sp, dt, (n, 3))
    Y, _ = run(sp, ctx, kern, A, X, k=3)
    assert_parity_multi(dt, Y, A, X, kern)


@pytest.mark.parametrize("k", [1, 2, 4, 8, 16, 32, 43])
@pytest.mark.parametrize("dt", [0, 1, 2, 3, 4, 5])
def test_panel_parity(sp, ctx, dt, k):
    """Panels of every width, whole 16-byte pieces of x or not, CSR and COO."""
    name = ["hub", "empties", "one", "exact"][(dt + k) % 4]
    n, m, row, col = _pattern(name, np.random.default_rng(k))
    A = _coo(sp, dt, n, m, row, col)
    for kern, ldx, ldy in (("CSR-nnz", k, k), ("COO-nnz", k + 1, k + 2)):
        X = _x(sp, dt, (m, ldx))
        plan = sp.Plan(ctx, kern, A)
        xd = sp.DeviceArray.from_numpy(ctx, X)
        yd = sp.DeviceArray(ctx, (n, ldy), X.dtype)
        yd.fill_bytes(0x5A)
        plan.spmm(k, xd.addr, ldx, yd.addr, ldy)
        ctx.sync()
        Y = yd.numpy()
        assert_parity_multi(dt, np.ascontiguousarray(Y[:, :k]), A, np.ascontiguousarray(X[:, :k]), f"{kern}/{name}/k{k}")
        assert np.all(Y[:, k:].view(np.uint8) == 0x5A)


@pytest.mark.parametrize("k", [2, 4, 8, 16, 32, 35])
@pytest.mark.parametrize("dt,rows,per", [(4, 3001, 33), (5, 3001, 33), (2, 40000, 5), (5, 9001, 4), (4, 33000, 33)])
def test_panel_even_rows(sp, ctx, dt, rows, per, k):
    """Even rows on both sides of the panel rule: row lengths, widths and sizes."""
    rng = np.random.default_rng(rows + k)
    row = np.repeat(np.arange(rows), per)
    A = _coo(sp, dt, rows, rows, row, rng.integers(0, rows, row.size))
    X = _x(sp, dt, (rows, k))
    Y, _ = run(sp, ctx, "CSR-nnz", A, X, k=k)
    assert_parity_multi(dt, Y, A, X, f"k{k}")


def test_wide_columns_too_far(sp, ctx):
    """Nearly every run would end early: the plan keeps row-ordered tiles."""
    rng = np.random.default_rng(2)
    n, m = 2000, 1 << 27
    row = np.concatenate([np.full(20000, 5), rng.integers(0, n, 20000)])
    A = _coo(sp, 0, n, m, row, rng.integers(0, m, row.size))
    x = _x(sp, 0, m)
    for kern in ("CSR-nnz", "COO-nnz"):
        y, plan = run(sp, ctx, kern, A, x)
        assert plan.info()["algo"] == sp.ALGO_SEGMENTED
        assert_parity(0, y, A, x, kern)


def test_wide_strides_and_knobs(sp, ctx):
    """One column of a wider panel; a memory cap or any knob keeps the kernels it had."""
    n, m, row, col = _pattern("hub", np.random.default_rng(1))
    A = _coo(sp, 4, n, m, row, col)
    X = _x(sp, 4, (m, 3))
    plan = sp.Plan(ctx, "CSR-nnz", A)
    xd = sp.DeviceArray.from_numpy(ctx, X)
    yd = sp.DeviceArray(ctx, (n, 2), np.float32)
    yd.fill_bytes(0)
    plan.spmm(1, xd.addr, 3, yd.addr, 2)
    ctx.sync()
    Y = yd.numpy()
    assert_parity(4, np.ascontiguousarray(Y[:, 0]), A, np.ascontiguousarray(X[:, 0]), "ldx 3")
    assert not Y[:, 1].any()
    one = sp.Plan(ctx, "CSR-nnz", A, sp.opts(mem_cap_bytes=1 << 20))
    assert one.info()["device_bytes"] <= 1 << 20 < plan.info()["device_bytes"]
    y, _ = run(sp, ctx, "CSR-nnz", A, np.ascontiguousarray(X[:, 1]), plan=one)
    assert_parity(4, y, A, np.ascontiguousarray(X[:, 1]), "memory cap")


def test_wide_in_batches(sp, ctx):
    """Wide plans of both shapes in one batch, with one and several right-hand sides."""
    mats, ks = [], [1, 1, 4, 1, 4, 43]
    for i, name in enumerate(["hub", "empties", "hub", "one", "exact", "one"]):
        mats.append(_coo(sp, 2, *_pattern(name, np.random.default_rng(i)), seed=i))
    plans = [sp.Plan(ctx, k, A) for k, A in zip(["CSR-nnz", "COO-nnz", "CSR-nnz", "COO-row", "COO-nnz", "CSR-row"], mats)]
    xs = [_x(sp, 2, (A.ncols, k)) for A, k in zip(mats, ks)]
    xd = [sp.DeviceArray.from_numpy(ctx, x) for x in xs]
    yd = [sp.DeviceArray(ctx, (A.nrows, k), np.int32) for A, k in zip(mats, ks)]
    batch = sp.Batch(ctx, plans, ks)
    for _ in range(3):
        for y in yd:
            y.fill_bytes(0x5A)
        batch.run([x.addr for x in xd], [y.addr for y in yd])
        ctx.sync()
        for A, x, y in zip(mats, xs, yd):
            assert_parity_multi(2, y.numpy(), A, x)
