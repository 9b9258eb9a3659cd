"""Where a conjugate-gradient solve (sp_cg) stops on the device: iterations that
the host has queued behind the last one change nothing, whatever iteration that
is and whatever ended the solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _diagonal(sp, d):
    i = np.arange(len(d), dtype=np.uint32)
    return sp.Coo.from_arrays(len(d), len(d), i, i, np.asarray(d, np.float64))


def _solve(sp, ctx, plan, b, **kw):
    bd, xd = sp.DeviceArray.from_numpy(ctx, b), sp.DeviceArray.from_numpy(ctx, np.zeros_like(b))
    it, res = plan.cg(bd.addr, xd.addr, **kw)
    return xd.numpy(), it, res


@pytest.mark.parametrize("n", [3, 700, 300000])
def test_queued_iterations_change_nothing(sp, ctx, n):
    """Stopped by rtol after `it` iterations, x has the bits of a solve with maxit = it, which
    queues none behind; `it` runs over odd and even numbers."""
    rng = np.random.default_rng(n)
    plan = sp.Plan(ctx, "CSR-nnz", _diagonal(sp, rng.uniform(1, 30, n)))
    b = rng.standard_normal(n)
    seen = set()
    for rtol in (0.7, 0.5, 0.3, 0.2, 0.1, 0.05, 1e-2, 1e-3, 1e-5):
        x, it, res = _solve(sp, ctx, plan, b, maxit=1000, rtol=rtol)
        xm, itm, resm = _solve(sp, ctx, plan, b, maxit=it, rtol=0.0)
        assert it == itm and res == resm <= rtol and np.array_equal(x, xm)
        seen.add(it % 2)
    assert seen == {0, 1}


def test_three_eigenvectors(sp, ctx):
    """b in the span of three eigenvectors: solved after three iterations, up to rounding."""
    d = np.resize([1.0, 2.0, 5.0], 4000)
    b = np.random.default_rng(2).standard_normal(4000)
    x, it, res = _solve(sp, ctx, sp.Plan(ctx, "CSR-nnz", _diagonal(sp, d)), b, maxit=50, rtol=1e-12)
    assert it == 3 and res <= 1e-12 and np.abs(x - b / d).max() <= 1e-11


def test_not_positive_definite(sp, ctx):
    """p'Ap <= 0 in the second iteration ends the solve with an error, and the plan solves again."""
    b = np.ones(2)
    plan = sp.Plan(ctx, "CSR-nnz", _diagonal(sp, [3.0, -1.0]))
    for _ in range(3):
        with pytest.raises(sp._lib.SparsePError):
            _solve(sp, ctx, plan, b, maxit=50, rtol=1e-12)
    good = sp.Plan(ctx, "CSR-nnz", _diagonal(sp, [3.0, 1.0]))
    x, it, _ = _solve(sp, ctx, good, b, maxit=50, rtol=1e-12)
    assert it == 2 and np.allclose(x, [1 / 3, 1.0], atol=1e-14)
