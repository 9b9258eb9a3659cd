"""The tuner's candidate points: every id's default first, and beside it, by
name, the kernels that the default takes on other matrices, so that each can be
timed whatever the automatic rules choose."""
import pytest


def _points(sp, A, kern):
    return [(p.opts.algo, p.opts.lanes_per_row, p.opts.items_per_lane, p.opts.vert, p.opts.lds_slice,
             p.opts.row_block_size) for p in sp.tune_space(A, sp.KID[kern])]


@pytest.mark.parametrize("kern,algo,ipt", [
    ("COO-row", 0, 4), ("COO-nnz-rgrn", 0, 4), ("COO-nnz", 0, 4), ("COO-nnz", 2, 0), ("CSR-nnz", 3, 8), ("CSR-row", 3, 16),
    ("CSR-nnz", 2, 8), ("DCSR", 1, 0), ("RBDCSR", 1, 0), ("BDCSR", 1, 0), ("RBDCSR", 3, 0), ("DCOO", 0, 8),
    ("RBDCOO", 0, 8), ("BDCOO", 0, 8), ("BCOO-block", 2, 0), ("BCOO-nnz", 2, 0), ("BCSR-nnz", 2, 0)])
def test_kernels_by_name(sp, kern, algo, ipt):
    A = sp.gen_uniform(3000, 3000, 20, 30, dtype=sp.F32, seed=1)
    pts = _points(sp, A, kern)
    assert pts[0] == (0, 0, 0, 0, 0, 4) and len(set(pts)) == len(pts)
    assert any(p[0] == algo and p[2] == ipt and p[3:] == (0, 0, 4) for p in pts[1:])


def test_row_kernels_by_name(sp):
    """The automatic row kernels' lanes: chunks of four entries, and whole rows below 16 entries."""
    pts = _points(sp, sp.gen_uniform(3000, 3000, 33, 33, dtype=sp.F32, seed=1), "CSR-nnz")
    assert any(p[:3] == (1, 16, 4) for p in pts)
    pts = _points(sp, sp.gen_uniform(3000, 3000, 5, 5, dtype=sp.F32, seed=1), "CSR-nnz")
    assert any(p[:3] == (1, 8, 0) for p in pts)
