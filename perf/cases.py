"""The work that programs have this library do, as cases that can be timed.

Each case is one use through the public entry points of `sparsep_amd.api`: a
matrix of one of the families that the tests and the bench generate, the plan
that a program keeps for it, and one call (or one solve) on device vectors.

ops
  spmv   y = A x through one of the 25 kernel ids (default options)
  spmm   Y = A X with k right-hand sides, X and Y row-major
  batch  many small problems of different k through one sp_batch (hipGraph)
  cg     conjugate gradient on a plan (an implicit diffusion step, FP64/FP32)
  grad   forward and backward of the variant selector's MLP on one mini-batch

matrix families (`matrix`): stencil5 (2D Laplacian), stencil27 (3D grid, 4
unknowns per point, periodic), rmat (power-law graph), uniform (2..64 entries
per row anywhere), banded (2..64 entries per row within 32 of the diagonal).
"""
import math

import numpy as np
import torch

import sparsep_amd.api as sp

DTYPES = {"i8": (sp.I8, torch.int8), "i16": (sp.I16, torch.int16), "i32": (sp.I32, torch.int32),
          "i64": (sp.I64, torch.int64), "f32": (sp.F32, torch.float32), "f64": (sp.F64, torch.float64)}
SIZE = {"i8": 1, "i16": 2, "i32": 4, "i64": 8, "f32": 4, "f64": 8}
RMAT_ABCD = (0.57, 0.19, 0.19, 0.05)
MLP = (64, 128, 128, 25)
BAND = 32


def listed():
    return [
        # the smallest call: a cache-resident 2D Laplacian in integers, where a launch's latency is the time
        {"name": "spmv_stencil5_csr_i32", "op": "spmv", "matrix": "stencil5", "n": 256, "kernel": "CSR-row",
         "dtype": "i32"},
        # the headline: one product with a power-law graph of 2^20 vertices and 2^24 edges
        {"name": "spmv_rmat20_csr_f32", "op": "spmv", "matrix": "rmat", "n": 20, "per_row": 16, "kernel": "CSR-nnz",
         "dtype": "f32"},
        # an ordinary graph in double precision, kept as coordinates (edge lists)
        {"name": "spmv_rmat18_coo_f64", "op": "spmv", "matrix": "rmat", "n": 18, "per_row": 16, "kernel": "COO-nnz",
         "dtype": "f64"},
        # one-byte data (quantised or counted), rectangular with odd sizes, rows of uneven length
        {"name": "spmv_uniform_csr_i8", "op": "spmv", "matrix": "uniform", "n": 300001, "cols": 200003,
         "kernel": "CSR-nnz", "dtype": "i8"},
        # a 3D simulation matrix with 4 unknowns per point in its own block format: the largest stream
        {"name": "spmv_stencil27_bcsr_f32", "op": "spmv", "matrix": "stencil27", "n": 64, "kernel": "BCSR-block",
         "dtype": "f32"},
        # the same kind of matrix in double precision as block coordinates, an odd grid
        {"name": "spmv_stencil27_bcoo_f64", "op": "spmv", "matrix": "stencil27", "n": 37, "kernel": "BCOO-nnz",
         "dtype": "f64"},
        # a 2D tiling (stripes of x, partial results merged), a band matrix of odd size
        {"name": "spmv_banded_rbdcsr_f32", "op": "spmv", "matrix": "banded", "n": 199999, "kernel": "RBDCSR",
         "dtype": "f32"},
        # several vectors at once on a graph: eight features per vertex
        {"name": "spmm8_rmat18_csr_f32", "op": "spmm", "matrix": "rmat", "n": 18, "per_row": 16, "kernel": "CSR-nnz",
         "dtype": "f32", "k": 8},
        # a block solver's panel of 32 vectors on the simulation matrix
        {"name": "spmm32_stencil27_bcsr_f32", "op": "spmm", "matrix": "stencil27", "n": 48, "kernel": "BCSR-block",
         "dtype": "f32", "k": 32},
        # many small uneven problems in one call
        {"name": "batch24_f32", "op": "batch", "problems": 24, "rows_max": 60000, "kernel": "CSR-nnz", "dtype": "f32"},
        # an iterative solve: one implicit diffusion step on a 512 x 512 grid, to 1e-10
        {"name": "cg_stencil5_f64", "op": "cg", "matrix": "stencil5", "n": 512, "kernel": "CSR-nnz", "dtype": "f64"},
        # one mini-batch of selector training: forward, loss and every gradient
        {"name": "grad_mlp_b64", "op": "grad", "batch": 64, "dtype": "f32"},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    op = rng.choices(["spmv", "spmm", "batch", "cg", "grad"], [10, 5, 2, 2, 2])[0]
    if op == "grad":
        return {"op": op, "batch": _log_int(rng, 16, 512), "dtype": "f32"}
    if op == "cg":
        return {"op": op, "matrix": "stencil5", "n": _log_int(rng, 60, 512), "kernel": rng.choice(["CSR-nnz", "CSR-row"]),
                "dtype": rng.choice(["f64", "f64", "f32"])}
    if op == "batch":
        return {"op": op, "problems": _log_int(rng, 4, 24), "rows_max": _log_int(rng, 4000, 60000),
                "kernel": "CSR-nnz", "dtype": rng.choice(["f32", "f32", "i16", "f64"])}
    c = {"op": op, "matrix": rng.choice(["stencil5", "rmat", "rmat", "uniform", "banded", "stencil27"])}
    if c["matrix"] == "stencil5":
        c["n"] = _log_int(rng, 100, 1500)
    elif c["matrix"] == "rmat":
        c["n"] = rng.randint(12, 19)
        c["per_row"] = rng.choice([8, 11, 16, 24])
    elif c["matrix"] == "stencil27":
        c["n"] = rng.randint(9, 40)
    else:
        c["n"] = _log_int(rng, 2000, 300000)
        if c["matrix"] == "uniform":
            c["cols"] = max(1000, int(c["n"] * rng.uniform(0.5, 1.5)))
    kernels = ["CSR-row", "CSR-nnz", "CSR-nnz", "COO-row", "COO-nnz-rgrn", "COO-nnz"]
    if op == "spmm":
        kernels = ["CSR-nnz", "CSR-nnz", "CSR-row", "COO-nnz"]
    elif c["matrix"] != "rmat":
        kernels += ["DCSR", "DCOO", "RBDCSR", "RBDCOO", "BDCSR", "BDCOO"]
    if c["matrix"] == "stencil27":
        kernels += ["BCSR-block", "BCSR-nnz"] * 2
        if op == "spmv":
            kernels += ["BCOO-block", "BCOO-nnz", "DBCSR", "RBDBCSR-block", "BDBCOO-nnz"]
    c["kernel"] = rng.choice(kernels)
    c["dtype"] = rng.choice(["f32", "f32", "f32", "f64", "f64", "i8", "i16", "i32", "i64"])
    if op == "spmm":
        c["k"] = rng.choice([2, 3, 4, 8, 8, 16, 32])
        while _rows(c) * c["k"] > 1 << 23:  # no wider a panel than the largest listed
            c["k"] //= 2
        if c["k"] < 2:
            c["op"] = "spmv"
            del c["k"]
    return c


# --------------------------------------------------------------------------
# matrices, made on the GPU from the seed
# --------------------------------------------------------------------------
def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    return g


def _rows(c):
    n = c["n"]
    return {"stencil5": n * n, "rmat": 1 << n if n < 31 else n, "stencil27": 4 * n ** 3}.get(c["matrix"], n)


def _cols(c):
    return c["cols"] if c["matrix"] == "uniform" else _rows(c)


def _nnz(c):
    """Entries of the matrix (their expected number where rows are random)."""
    n = c["n"]
    if c["matrix"] == "stencil5":
        return 5 * n * n - 4 * n
    if c["matrix"] == "rmat":
        return c["per_row"] << n
    if c["matrix"] == "stencil27":
        return 27 * 16 * n ** 3
    return 33 * n


def _values(count, dtype, g):
    if dtype[0] == "i":  # small whole numbers, -4 .. 4
        return torch.randint(-4, 5, (count,), generator=g, device="cuda", dtype=torch.int32).to(DTYPES[dtype][1])
    return torch.rand(count, generator=g, device="cuda", dtype=DTYPES[dtype][1]) * 2 - 1


def _pattern(c, g):
    """Row and column indices (int64) in row order."""
    n, m = _rows(c), c["matrix"]
    dev = {"device": "cuda"}
    if m == "stencil5":
        side = c["n"]
        v = torch.arange(n, **dev)[:, None]
        d = torch.tensor([-side, -1, 0, 1, side], **dev)
        x = v % side + torch.tensor([0, -1, 0, 1, 0], **dev)
        col = v + d
        ok = (x >= 0) & (x < side) & (col >= 0) & (col < n)
        return v.expand(-1, 5)[ok], col[ok]
    if m == "stencil27":
        side = c["n"]
        v = torch.arange(side ** 3, **dev)
        x, y, z = v % side, v // side % side, v // (side * side)
        o = torch.tensor([-1, 0, 1], **dev)
        nb = (((z[:, None] + o) % side)[:, :, None, None] * side + ((y[:, None] + o) % side)[:, None, :, None]) * side \
            + ((x[:, None] + o) % side)[:, None, None, :]
        nb = nb.reshape(-1, 27).sort(1)[0]
        col = (nb[:, None, :, None] * 4 + torch.arange(4, **dev)).expand(-1, 4, 27, 4)
        row = (v[:, None] * 4 + torch.arange(4, **dev))[:, :, None].expand(-1, 4, 108)
        return row.reshape(-1), col.reshape(-1)
    if m == "banded":
        keep = torch.rand(n, generator=g, **dev) * (62 / 65) + 2 / 65  # 2 .. 64 of the 65 columns of the window
        row, at = (torch.rand(n, 2 * BAND + 1, generator=g, **dev) < keep[:, None]).nonzero(as_tuple=True)
        col = row + at - BAND
        ok = (col >= 0) & (col < n)
        return row[ok], col[ok]
    if m == "uniform":
        row = torch.repeat_interleave(torch.arange(n, **dev), torch.randint(2, 65, (n,), generator=g, **dev))
        key = row * c["cols"] + torch.randint(0, c["cols"], row.shape, generator=g, **dev)
        key = torch.unique(key)
        return key // c["cols"], key % c["cols"]
    a, b, cc, _ = RMAT_ABCD
    scale, want = c["n"], _nnz(c)
    key = torch.empty(0, dtype=torch.int64, **dev)
    while key.numel() < want:
        count = int((want - key.numel()) * 1.3) + 1000
        row = torch.zeros(count, dtype=torch.int64, **dev)
        col = torch.zeros(count, dtype=torch.int64, **dev)
        for _ in range(scale):
            u = torch.rand(count, generator=g, **dev)
            low = u >= a + b
            row = row * 2 + low
            col = col * 2 + (torch.where(low, u >= a + b + cc, u >= a))
        key = torch.unique(torch.cat([key, (row << scale) + col]))
    if key.numel() > want:  # distinct edges, as many as asked for
        key = key[torch.randperm(key.numel(), generator=g, **dev)[:want].sort()[0]]
    return key >> scale, key & ((1 << scale) - 1)


def _matrix(c, seed):
    """Row indices, column indices and values on the GPU."""
    g = _gen(seed)
    row, col = _pattern(c, g)
    if c["op"] == "cg":  # one step of implicit diffusion: the identity plus the Laplacian
        val = torch.where(row == col, 5.0, -1.0).to(DTYPES[c["dtype"]][1])
    else:
        val = _values(row.numel(), c["dtype"], g)
    return row, col, val, g


def _coo(c, row, col, val):
    return sp.Coo.from_arrays(_rows(c), _cols(c), row.to(torch.int32).cpu().numpy().view(np.uint32),
                              col.to(torch.int32).cpu().numpy().view(np.uint32), val.cpu().numpy())


def _product(c, row, col, val, x):
    """A x in 64 bits: whole numbers modulo their type's size, real numbers in double precision."""
    wide = torch.int64 if c["dtype"][0] == "i" else torch.float64
    y = torch.zeros((_rows(c),) + tuple(x.shape[1:]), dtype=wide, device="cuda")
    step = max(1, (1 << 28) // max(1, x[0].numel()))
    for i in range(0, row.numel(), step):
        p = val[i:i + step].to(wide)
        xs = x[col[i:i + step]].to(wide)
        y.index_add_(0, row[i:i + step], p * xs if x.dim() == 1 else p[:, None] * xs)
    return y.to(DTYPES[c["dtype"]][1]) if wide == torch.int64 else y


_ctx = []


def _context():
    """The program's one context (a stream on the device)."""
    if not _ctx:
        _ctx.append(sp.Context(0))
    return _ctx[0]


def _problems(c, seed):
    """The members of a batch: their shapes follow from the case, their entries from the seed."""
    r = np.random.default_rng(c["problems"] * 1000003 + c["rows_max"])
    for i in range(c["problems"]):
        n = int(math.exp(r.uniform(math.log(1000), math.log(c["rows_max"]))))
        p = {"op": "spmm", "dtype": c["dtype"], "kernel": c["kernel"], "k": [1, 4, 8, 32][i % 4]}
        if i % 3 == 2:
            p.update(matrix="rmat", n=max(10, int(math.log2(n))), per_row=16)
        elif i % 3 == 1:
            p.update(matrix="banded", n=n)
        else:
            p.update(matrix="uniform", n=n, cols=n)
        yield p, seed * 100 + i


def _vectors(c, g):
    k = c.get("k", 1)
    x = _values(_cols(c) * k, c["dtype"], g)
    return x.view(-1, k) if c["op"] == "spmm" else x


def _mlp_inputs(c, seed):
    """Standardised features, log2 slowdowns clipped to 0 .. 6, the mask of timed variants, and He-sized weights."""
    g = torch.Generator()
    g.manual_seed(seed)
    i, h1, h2, o = MLP
    x = torch.randn(c["batch"], i, generator=g)
    t = torch.randn(c["batch"], o, generator=g).abs_().mul_(2).clamp_(max=6)
    m = (torch.rand(c["batch"], o, generator=g) < 0.9).float()
    p = []
    for a, b in ((i, h1), (h1, h2), (h2, o)):
        p += [(torch.rand(b * a, generator=g) * 2 - 1) * math.sqrt(6 / a), torch.randn(b, generator=g) * 0.05]
    return x, t, m, torch.cat(p)


# --------------------------------------------------------------------------
# one case
# --------------------------------------------------------------------------
def prepare(case, seed):
    c, ctx, op = case, _context(), case["op"]
    if op == "grad":
        x, t, m, p = _mlp_inputs(c, seed)
        mlp = sp.Mlp(ctx, MLP, seed=5)
        mlp.set_params(p.numpy())
        return {"op": op, "mlp": mlp, "x": x.numpy(), "t": t.numpy(), "m": m.numpy()}
    if op == "batch":
        plans, ks, xs, ys = [], [], [], []
        for p, s in _problems(c, seed):
            row, col, val, g = _matrix(p, s)
            plans.append(sp.Plan(ctx, p["kernel"], _coo(p, row, col, val)))
            ks.append(p["k"])
            xs.append(_vectors(p, g))
            ys.append(torch.zeros(_rows(p), p["k"], dtype=xs[-1].dtype, device="cuda"))
        torch.cuda.synchronize()
        return {"op": op, "batch": sp.Batch(ctx, plans, ks), "xs": xs, "ys": ys,
                "xp": [x.data_ptr() for x in xs], "yp": [y.data_ptr() for y in ys]}
    row, col, val, g = _matrix(c, seed)
    plan = sp.Plan(ctx, c["kernel"], _coo(c, row, col, val))
    x = _vectors(c, g)
    if op == "cg":  # the right-hand side of a known solution, and a zero start
        b = _product(c, row, col, val, x).to(x.dtype)
        x, y = b, torch.zeros_like(b)
    else:
        y = torch.zeros((_rows(c),) + tuple(x.shape[1:]), dtype=x.dtype, device="cuda")
    torch.cuda.synchronize()
    return {"op": op, "plan": plan, "x": x, "y": y, "k": c.get("k", 1), "rtol": 1e-10 if c["dtype"] == "f64" else 1e-5}


def run(s):
    op, k = s["op"], s.get("k", 1)
    if op == "spmv":
        s["plan"].spmv(s["x"].data_ptr(), s["y"].data_ptr())
        return s["y"]
    if op == "spmm":
        s["plan"].spmm(k, s["x"].data_ptr(), k, s["y"].data_ptr(), k)
        return s["y"]
    if op == "batch":
        s["batch"].run(s["xp"], s["yp"])
        return s["ys"]
    if op == "cg":
        s["y"].zero_()
        s["plan"].cg(s["x"].data_ptr(), s["y"].data_ptr(), maxit=500, rtol=s["rtol"])
        return s["y"]
    loss, grad = s["mlp"].loss_grad(s["x"], s["t"], s["m"])
    return {"loss": loss, "grad": grad}


def exact(case, seed):
    c, op = case, case["op"]
    if op == "grad":
        x, t, m, p = (v.double() for v in _mlp_inputs(c, seed))
        i, h1, h2, o = MLP
        w, at = [], 0
        for a, b in ((i, h1), (h1, h2), (h2, o)):  # weights are used in bfloat16, biases as they are
            w.append(p[at:at + a * b].float().bfloat16().double().view(b, a).requires_grad_())
            w.append(p[at + a * b:at + a * b + b].clone().requires_grad_())
            at += a * b + b
        a1 = (x @ w[0].T + w[1]).relu()
        a2 = (a1 @ w[2].T + w[3]).relu()
        loss = (((a2 @ w[4].T + w[5]) - t) * m).square().sum() / t.numel()
        loss.backward()
        return {"loss": loss.item(), "grad": torch.cat([v.grad.reshape(-1) for v in w])}
    if op == "batch":
        out = []
        for p, s in _problems(c, seed):
            row, col, val, g = _matrix(p, s)
            out.append(_product(p, row, col, val, _vectors(p, g)))
        return out
    row, col, val, g = _matrix(c, seed)
    x = _vectors(c, g)
    return x.double() if op == "cg" else _product(c, row, col, val, x)  # cg: the solution that b was made from


def _format_bytes(c):
    """The matrix once, in the format that the kernel id names."""
    s, n, nnz, name = SIZE[c["dtype"]], _rows(c), _nnz(c), c["kernel"]
    if "BCSR" in name:  # 4 x 4 blocks of the 4 unknowns per point, all full
        return nnz // 16 * (16 * s + 4) + (n // 4 + 1) * 4
    if "BCOO" in name:
        return nnz // 16 * (16 * s + 8)
    return nnz * (s + 8) if "COO" in name else nnz * (s + 4) + (n + 1) * 4


def work(case):
    c, op = case, case["op"]
    if op == "grad":
        i, h1, h2, o = MLP
        p, b = i * h1 + h1 * h2 + h2 * o, c["batch"]
        return {"bytes": 4 * (2 * p + b * (i + 2 * o)), "flops": 2 * b * (3 * p - i * h1)}
    if op == "batch":
        each = [work(p) for p, _ in _problems(c, 0)]
        return {q: sum(e[q] for e in each) for q in ("bytes", "flops")}
    s, k, n = SIZE[c["dtype"]], c.get("k", 1), _rows(c)
    one = {"bytes": _format_bytes(c) + (n + _cols(c)) * k * s, "flops": 2 * _nnz(c) * k}
    if op == "cg":  # about 35 iterations to 1e-10, 17 to 1e-5: the product, three updates and two dot products each
        it = 35 if c["dtype"] == "f64" else 17
        return {"bytes": it * (one["bytes"] + 6 * n * s), "flops": it * (one["flops"] + 10 * n)}
    return one
