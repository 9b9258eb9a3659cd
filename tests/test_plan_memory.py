"""Device memory of plans, on a device that is simulated in host memory
(fake_device.c): a second layout that has no room is left out, so a matrix that
fits once gets its plan, and a plan frees what it does not keep."""
import os
import shutil
import subprocess
import sys

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))

PLANS = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_limit.argtypes = [ctypes.c_size_t]
fake.fake_live.restype = ctypes.c_size_t
import numpy as np
import sparsep_amd.api as sp
NONE = 2 ** 64 - 1
kern, matrix, dt, k = sys.argv[2], sys.argv[3], int(sys.argv[4]), int(sys.argv[5])
ctx = sp.Context(0)
if matrix == "rmat":
    A = sp.gen_rmat(13, 100000, dtype=dt, seed=1)
elif matrix == "even":
    A = sp.gen_banded(40000, 32, 20, 40, dtype=dt, seed=2)
elif matrix == "blocks":
    A = sp.gen_stencil27(34, 4, True, dt, seed=3)
else:  # "gaps": the second of two stripes has more rows per entry than a wide tile takes
    n = 400000
    row = np.concatenate([np.repeat(np.arange(n), 3), np.arange(0, n, 20)])
    col = np.concatenate([np.tile(np.arange(3), n), np.full(n // 20, n - 1)])
    o = np.lexsort((col, row))
    A = sp.Coo.from_arrays(n, n, row[o].astype(np.uint32), col[o].astype(np.uint32), np.ones(o.size, sp.NP_DTYPE[dt]))
x, y = 64, 64  # (kernels do not run)


def product(plan):
    if k == 1:
        plan.spmv(x, y)
    else:
        plan.spmm(k, x, k, y, k)


base = fake.fake_live()
plan = sp.Plan(ctx, kern, A, sp.opts(mem_cap_bytes=1 << 40))  # (a cap: one layout)
product(plan)
need = fake.fake_live() - base
once = plan.info()
del plan
plan = sp.Plan(ctx, kern, A)
product(plan)
full = fake.fake_live() - base
assert full == plan.info()["device_bytes"], (full, plan.info())
both = plan.info()
del plan
assert fake.fake_live() == base
if k == 1 and dt >= 4 and A.nrows == A.ncols:  # a solve's vectors are kept, and counted
    plan = sp.Plan(ctx, kern, A)
    product(plan)
    for _ in range(2):
        try:
            plan.cg(x, y, maxit=3)
        except sp._lib.SparsePError:
            pass
        kept = fake.fake_live() - base - full
        assert kept >= 3 * A.nrows * sp.NP_DTYPE[dt]().itemsize
        assert fake.fake_live() - base == plan.info()["device_bytes"]
    del plan
    assert fake.fake_live() == base
    plan = sp.Plan(ctx, kern, A)
    product(plan)
    fake.fake_limit(fake.fake_live())
    for _ in range(2):  # no room for them: an error of its own, and the plan still multiplies
        try:
            plan.cg(x, y, maxit=3)
            raise SystemExit("a solve without memory")
        except sp._lib.SparsePError as e:
            assert e.rc == -2
        product(plan)
    assert plan.info()["device_bytes"] == full
    del plan
    fake.fake_limit(NONE)
print("need", need, "full", full, "algo", once["algo"], both["algo"], flush=True)
assert matrix == "gaps" or full > need
for part in range(9):
    limit = base + need + (full - need) * part // 8
    fake.fake_limit(limit)
    plan = sp.Plan(ctx, kern, A)
    product(plan)
    i = plan.info()
    assert fake.fake_live() - base == i["device_bytes"] <= limit - base
    if part == 0:
        assert (i["algo"], i["launches"]) == (once["algo"], once["launches"])
    if part == 8:
        assert (i["algo"], i["launches"]) == (both["algo"], both["launches"])
    del plan
    fake.fake_limit(NONE)
    assert fake.fake_live() == base
if matrix == "gaps":
    assert both["algo"] == once["algo"] and full == need, "the parts of a layout that was given up are kept"
print("ok")
"""


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    if not shutil.which("gcc") or not os.path.exists("/opt/rocm/include/hip/hip_runtime_api.h"):
        pytest.skip("no C compiler or no HIP headers")
    so = str(tmp_path_factory.mktemp("fake") / "fake_device.so")
    subprocess.run(["gcc", "-shared", "-fPIC", "-O1", "-w", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include",
                    os.path.join(HERE, "fake_device.c"), "-o", so], check=True)
    return so


BCOO_ROUTES = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import sparsep_amd.api as sp
ctx = sp.Context(0)
for dt, g, rc, algo in [(sp.F32, 32, (4, 4), sp.ALGO_VECTOR), (sp.F32, 33, (4, 4), sp.ALGO_SEGMENTED),
                        (sp.I32, 25, (2, 4), sp.ALGO_VECTOR), (sp.I32, 26, (2, 4), sp.ALGO_SEGMENTED),
                        (sp.F64, 25, (2, 2), sp.ALGO_VECTOR), (sp.F64, 26, (2, 2), sp.ALGO_SEGMENTED),
                        (sp.F64, 33, (4, 4), sp.ALGO_VECTOR), (sp.F64, 33, (4, 2), sp.ALGO_VECTOR)]:
    A = sp.gen_stencil27(g, 4, True, dt, seed=3)
    i = sp.Plan(ctx, "BCOO-nnz", A, sp.opts(row_block_size=rc[0], col_block_size=rc[1])).info()
    assert i["algo"] == algo, (dt, g, rc, i)
print("ok")
"""


def test_bcoo_block_rows_where_they_are_faster(fake):
    r = subprocess.run([sys.executable, "-c", BCOO_ROUTES, fake], cwd=os.path.dirname(HERE), capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


TILES = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import sparsep_amd.api as sp
ctx = sp.Context(0)
for dt, nnz, small in [(sp.F64, 2800000, True), (sp.F64, 3200000, False), (sp.F32, 2800000, True), (sp.F32, 3200000, False)]:
    n = nnz // 20
    row = np.repeat(np.arange(n, dtype=np.uint32), 20)
    col = np.sort(np.random.default_rng(1).integers(0, n, (n, 20)), axis=1).ravel().astype(np.uint32)
    i = sp.Plan(ctx, "COO-nnz", sp.Coo.from_arrays(n, n, row, col, np.ones(row.size, sp.NP_DTYPE[dt]))).info()
    assert i["algo"] == sp.ALGO_SEGMENTED_SORTED and (i["ntiles"] > 600) == small, (dt, nnz, i)
    # threads and entries per thread; merge tiles of the same name report no lanes, and what is
    # reported can be asked for
    assert (i["lanes_per_row"], i["items_per_lane"]) == ((512 if dt == sp.F32 else 256, 8) if small
                                                         else (1024, 16 if dt == sp.F32 else 8))
    A = sp.Coo.from_arrays(n, n, row, col, np.ones(row.size, sp.NP_DTYPE[dt]))
    for kern in ("CSR-nnz", "COO-nnz"):
        j = sp.Plan(ctx, kern, A, sp.opts(algo=i["algo"], items_per_lane=i["items_per_lane"],
                                          lanes_per_row=i["lanes_per_row"] if kern == "COO-nnz" else 0)).info()
        assert j["algo"] == i["algo"] and j["lanes_per_row"] == 0 and j["items_per_lane"] == i["items_per_lane"], j
print("ok")
"""


def test_wide_tile_sizes(fake):
    """Scattered columns: small tiles up to 3M entries, for either size of sums."""
    r = subprocess.run([sys.executable, "-c", TILES, fake], cwd=os.path.dirname(HERE), capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


CSR_ROUTES = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
import numpy as np
import sparsep_amd.api as sp
ctx = sp.Context(0)


def matrix(lens, local, dt):
    rng = np.random.default_rng(1)
    n = len(lens)
    m = n + 80 if local else n
    row = np.repeat(np.arange(n), lens)
    key = np.sort(row * m + (row + rng.integers(0, 80, row.size) if local else rng.integers(0, m, row.size)))
    return sp.Coo.from_arrays(n, m, (key // m).astype(np.uint32), (key % m).astype(np.uint32),
                              np.ones(key.size, sp.NP_DTYPE[dt]))


def spread(lo, hi, n):
    return np.random.default_rng(2).integers(lo, hi + 1, n)


fake.fake_launches.restype = ctypes.c_size_t
for lens, local, dt, k, launches in [  # the row kernels take one launch, panels two
        (np.full(18000, 17), True, sp.F32, 2, 1), (np.full(18000, 17), False, sp.F64, 4, 1),
        (np.full(130000, 17), True, sp.F64, 2, 2), (np.full(18000, 17), True, sp.F32, 16, 2),
        (np.full(130000, 17), True, sp.F32, 8, 1), (np.full(130000, 17), False, sp.F32, 8, 2),
        (spread(2, 64, 2500), True, sp.F32, 4, 1), (spread(2, 64, 3500), True, sp.F32, 4, 2),
        (spread(2, 64, 14000), True, sp.F32, 2, 1), (spread(2, 64, 18000), True, sp.F32, 2, 2),
        (np.full(35000, 63), True, sp.F32, 16, 2), (np.full(45000, 63), True, sp.F32, 16, 1),
        (np.full(100000, 12), True, sp.F64, 32, 1), (np.full(100000, 12), True, sp.F64, 16, 2),
        (np.full(40000, 33), True, sp.F32, 32, 1), (np.full(30000, 33), True, sp.F32, 32, 2)]:
    plan = sp.Plan(ctx, "CSR-row", matrix(lens, local, dt))
    n = fake.fake_launches()
    plan.spmm(k, 64, k, 64, k)
    assert fake.fake_launches() - n == launches, (lens[:4], len(lens), local, dt, k, fake.fake_launches() - n)
for lens, local, dt, ks, groups in [  # batch members of one width share panels, whatever their sizes
        ([spread(2, 64, 1000), spread(2, 64, 9000)], True, sp.F32, [4, 4], 1),
        ([np.full(600, 33), spread(2, 64, 9000)], False, sp.F64, [2, 2], 1),
        ([np.full(2000, 33), np.full(9000, 33)], False, sp.F32, [8, 8], 1),
        ([np.full(2000, 33), spread(2, 64, 9000)], True, sp.F32, [8, 8], 2),
        ([spread(2, 64, 1000), spread(2, 64, 9000)], True, sp.F32, [4, 8], 2)]:
    plans = [sp.Plan(ctx, "CSR-nnz", matrix(n, local, dt)) for n in lens]
    batch = sp.Batch(ctx, plans, ks, graph=False)
    assert batch.info()["groups"] == groups, (dt, ks, local, batch.info())
    n = fake.fake_launches()
    batch.run([64] * 2, [64] * 2)
    assert fake.fake_launches() - n == (3 if len(lens[0]) == 2000 and local else 2 * groups), (dt, ks, local)
ROWS, WIDE = sp.ALGO_VECTOR, sp.ALGO_SEGMENTED_SORTED
for lens, local, dt, algo in [
        (np.full(100000, 17), True, sp.F32, ROWS), (np.full(290000, 17), True, sp.F32, WIDE),
        (np.full(60000, 27), True, sp.F64, ROWS), (np.full(20000, 16), True, sp.F32, WIDE),
        (np.full(30000, 33), False, sp.F32, ROWS), (np.full(60000, 33), False, sp.F32, WIDE),
        (np.full(100000, 17), False, sp.F64, ROWS), (np.full(120000, 17), False, sp.F64, WIDE),
        (np.full(4000, 63), True, sp.I8, ROWS), (np.full(5000, 63), True, sp.I8, WIDE),
        (spread(2, 64, 10000), True, sp.F32, ROWS), (spread(2, 64, 20000), True, sp.F32, WIDE),
        (np.full(250000, 5), True, sp.F32, ROWS), (np.full(300000, 5), True, sp.F32, WIDE),
        (np.full(110000, 15), True, sp.F32, ROWS), (np.full(130000, 15), True, sp.F32, WIDE),
        (np.full(160000, 8), False, sp.F32, ROWS), (np.full(220000, 8), False, sp.F32, WIDE),
        (np.full(300000, 8), False, sp.F64, ROWS)]:
    i = sp.Plan(ctx, "CSR-nnz", matrix(lens, local, dt)).info()
    assert i["algo"] == algo, (lens[:4], len(lens), local, dt, i)
for lens, local, algo in [(np.full(300000, 5), True, ROWS), (np.full(530000, 5), True, WIDE),
                          (np.full(300000, 5), False, WIDE), (np.full(70000, 17), True, WIDE)]:
    i = sp.Plan(ctx, "RBDCSR", matrix(lens, local, sp.F32)).info()
    assert i["algo"] == algo, ("RBDCSR", lens[:4], len(lens), local, i)
print("ok")
"""


def test_even_rows_take_wide_tiles_where_they_are_faster(fake):
    r = subprocess.run([sys.executable, "-c", CSR_ROUTES, fake], cwd=os.path.dirname(HERE), capture_output=True,
                       text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


MLP = r"""
import ctypes, sys
fake = ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)
fake.fake_pinned.restype = ctypes.c_size_t
import numpy as np
import sparsep_amd.api as sp
mlp = sp.Mlp(sp.Context(0), (64, 128, 128, 25))
X, T = np.zeros((4000, 64), np.float32), np.zeros((4000, 25), np.float32)
mlp.predict(X)
assert fake.fake_pinned() == 0, "prediction pins host memory"
mlp.train(X, T, epochs=1, batch=64)
out = fake.fake_pinned()
assert 0 < out <= 4 * (mlp.nparams + 64 * 25 // 256 + 2), "training needs room for a gradient and its loss"
mlp.loss_grad(X[:64], T[:64])
both = fake.fake_pinned()
assert both == out + 64 * (64 + 2 * 25) * 4
mlp.predict(X)
mlp.loss_grad(X[:1], T[:1])
assert fake.fake_pinned() == both
mlp.loss_grad(X, T)
del mlp
assert fake.fake_pinned() == 0
print("ok")
"""


def test_selector_pins_only_for_gradients(fake):
    r = subprocess.run([sys.executable, "-c", MLP, fake], cwd=os.path.dirname(HERE), capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr


@pytest.mark.parametrize("kern,matrix,dt,k", [
    ("CSR-nnz", "rmat", 4, 1), ("CSR-nnz", "rmat", 3, 8), ("CSR-row", "even", 4, 1), ("CSR-row", "even", 2, 4),
    ("COO-nnz", "rmat", 5, 1), ("COO-nnz", "rmat", 0, 32), ("COO-row", "even", 4, 2),
    ("RBDCSR", "even", 4, 1), ("BDCOO", "even", 5, 1), ("DCOO", "even", 2, 3),
    ("BCOO-nnz", "blocks", 4, 1), ("BCOO-block", "blocks", 2, 8), ("RBDCOO", "gaps", 0, 1)])
def test_second_layouts_only_where_they_fit(fake, kern, matrix, dt, k):
    r = subprocess.run([sys.executable, "-c", PLANS, fake, kern, matrix, str(dt), str(k)], cwd=os.path.dirname(HERE),
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0 and r.stdout.endswith("ok\n"), r.stdout + r.stderr
