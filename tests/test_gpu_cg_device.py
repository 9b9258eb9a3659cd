"""Conjugate gradient whose scalars stay on the device (sp_cg): sizes around
the reduction grid, where it stops, what it reports, and plans used by
several threads.  The reference is the same recurrence in float64 numpy."""
import threading

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _tridiag(sp, dt, n):
    i = np.arange(n)
    row = np.concatenate([i, i[1:], i[:-1]])
    col = np.concatenate([i, i[:-1], i[1:]])
    val = np.concatenate([np.full(n, 4.0), np.full(2 * (n - 1), -1.0)])
    o = np.lexsort((col, row))
    return sp.Coo.from_arrays(n, n, row[o].astype(np.uint32), col[o].astype(np.uint32), val[o].astype(sp.NP_DTYPE[dt]))


def _mul(v):
    y = 4.0 * v
    y[1:] -= v[:-1]
    y[:-1] -= v[1:]
    return y


def _cg(b, maxit, rtol):
    x, r = np.zeros_like(b), b.copy()
    p, rr, it = r.copy(), r @ r, 0
    bn = np.sqrt(b @ b) or 1.0
    while it < maxit and np.sqrt(rr) / bn > rtol:
        q = _mul(p)
        a = rr / (p @ q)
        x += a * p
        r -= a * q
        r1 = r @ r
        p = r + (r1 / rr) * p
        rr, it = r1, it + 1
    return x, it, np.sqrt(rr) / bn


def _solve(sp, ctx, plan, b, x0=None, **kw):
    bd = sp.DeviceArray.from_numpy(ctx, b)
    xd = sp.DeviceArray.from_numpy(ctx, np.zeros_like(b) if x0 is None else x0)
    it, res = plan.cg(bd.addr, xd.addr, **kw)
    return xd.numpy(), it, res


@pytest.mark.parametrize("n", [1, 2, 255, 257, 1024, 262144, 262145, 600001])
def test_cg_sizes(sp, ctx, n):
    b = np.random.default_rng(n).standard_normal(n)
    plan = sp.Plan(ctx, "CSR-nnz", _tridiag(sp, 5, n))
    for maxit in (0, 1, 3, 200):
        want, itw, resw = _cg(b, maxit, 1e-9)
        x, it, res = _solve(sp, ctx, plan, b, maxit=maxit, rtol=1e-9)
        assert it == itw and abs(res - resw) <= 1e-6 * resw + 1e-15, (maxit, it, itw, res, resw)
        assert np.linalg.norm(x - want) <= 1e-12 * np.linalg.norm(b)


def test_cg_stops(sp, ctx):
    n = 5000
    plan = sp.Plan(ctx, "CSR-row", _tridiag(sp, 5, n))
    xt = np.random.default_rng(1).standard_normal(n)
    b = _mul(xt)
    x, it, res = _solve(sp, ctx, plan, b, x0=xt, maxit=50, rtol=1e-9)  # starts solved
    assert it == 0 and np.array_equal(x, xt)
    x, it, res = _solve(sp, ctx, plan, np.zeros(n), maxit=50, rtol=1e-9)
    assert it == 0 and res == 0 and not x.any()
    # b in the span of three eigenvectors and rtol 0: p.A p reaches zero or the limit holds
    x, it, _ = _solve(sp, ctx, plan, b, maxit=7, rtol=0.0)
    assert it == 7


def test_cg_threads_and_memory_cap(sp, ctx):
    """Solves on one plan from several threads, and on a plan that keeps no vectors."""
    n = 20000
    A = _tridiag(sp, 5, n)
    plans = [sp.Plan(ctx, "CSR-nnz", A), sp.Plan(ctx, "CSR-nnz", A, sp.opts(mem_cap_bytes=8 << 20))]
    bs = [np.random.default_rng(i).standard_normal(n) for i in range(4)]
    for plan in plans:
        got = [None] * 4

        def work(i):
            got[i] = _solve(sp, ctx, plan, bs[i], maxit=100, rtol=1e-11)

        ts = [threading.Thread(target=work, args=(i,)) for i in range(4)]
        for t in ts:
            t.start()
        for t in ts:
            t.join()
        for b, (x, it, res) in zip(bs, got):
            assert res <= 1e-11
            assert np.linalg.norm(_mul(x) - b) <= 1e-10 * np.linalg.norm(b)
