"""Products and solves on one plan from several threads at once: every result
has the bits of the same call made alone, also where a product is several
launches that hand over carries or partial vectors (wide tiles, merge tiles,
panels, 2D tilings)."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu
THREADS, ROUNDS = 4, 25


def _banded(sp, dt, n, per):
    """Symmetric, positive definite, 2 per + 1 entries per row (wide tiles from 3.7M entries on)."""
    i = np.arange(n)
    row, col, val = [i], [i], [np.full(n, 2.0 * per + 1)]
    for d in range(1, per + 1):
        row += [i[d:], i[:-d]]
        col += [i[:-d], i[d:]]
        val += [np.full(n - d, -1.0)] * 2
    row, col, val = (np.concatenate(v) for v in (row, col, val))
    o = np.lexsort((col, row))
    return sp.Coo.from_arrays(n, n, row[o].astype(np.uint32), col[o].astype(np.uint32), val[o].astype(sp.NP_DTYPE[dt]))


def _together(work):
    errors = []

    def guarded(i):
        try:
            work(i)
        except BaseException as e:  # shown by the caller
            errors.append(e)

    ts = [threading.Thread(target=guarded, args=(i,)) for i in range(THREADS)]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    if errors:
        raise errors[0]


@pytest.mark.parametrize("kern,k,algo", [("CSR-nnz", 1, 0), ("COO-nnz", 1, 0), ("CSR-nnz", 8, 0), ("CSR-nnz", 1, 2),
                                         ("RBDCSR", 1, 0), ("DCOO", 2, 0)])
def test_products_on_one_plan(sp, ctx, kern, k, algo):
    A = _banded(sp, 5, 70001, 12) if "D" in kern else sp.gen_rmat(15, 400000, dtype=sp.F64, seed=4)
    plan = sp.Plan(ctx, kern, A, sp.opts(algo=algo))
    rng = np.random.default_rng(k)
    xs = [sp.DeviceArray.from_numpy(ctx, rng.uniform(-1, 1, (A.ncols, k))) for _ in range(THREADS)]
    ys = [[sp.DeviceArray(ctx, (A.nrows, k), np.float64) for _ in range(2)] for _ in range(THREADS)]
    want = []
    for x, y in zip(xs, ys):
        plan.spmm(k, x.addr, k, y[0].addr, k)
        ctx.sync()
        want.append(y[0].numpy())
    got = [None] * THREADS

    def work(i):
        bad = 0
        for r in range(ROUNDS):
            for y in ys[i]:
                plan.spmm(k, xs[i].addr, k, y.addr, k)
            if r % 8 == 7:
                bad += sum(not np.array_equal(y.numpy(), want[i]) for y in ys[i])
        ctx.sync()
        got[i] = bad + sum(not np.array_equal(y.numpy(), want[i]) for y in ys[i])

    _together(work)
    assert got == [0] * THREADS


@pytest.mark.parametrize("kern", ["CSR-nnz", "RBDCSR"])
def test_solves_on_one_plan(sp, ctx, kern):
    A = _banded(sp, 5, 150001, 12)
    plan = sp.Plan(ctx, kern, A)
    assert plan.info()["algo"] == sp.ALGO_SEGMENTED_SORTED and plan.info()["launches"] >= 2
    bs = [sp.DeviceArray.from_numpy(ctx, np.random.default_rng(i).standard_normal(A.nrows)) for i in range(THREADS)]

    def solve(i):
        x = sp.DeviceArray.from_numpy(ctx, np.zeros(A.nrows))
        it, res = plan.cg(bs[i].addr, x.addr, maxit=60, rtol=1e-11)
        return x.numpy(), it, res

    want = [solve(i) for i in range(THREADS)]
    got = [None] * THREADS

    def work(i):
        got[i] = [solve(i) for _ in range(5)]

    _together(work)
    for w, g in zip(want, got):
        for x, it, res in g:
            assert it == w[1] and res == w[2] and np.array_equal(x, w[0])
