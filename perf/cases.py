"""The work that a program built on cumat_amd has it do, as measurable cases.

Every case is one pass through the public Python entry points on data that is
already on the GPU. The families, and what they stand for:

  cwise        one assignment of a component-wise expression: the update and
               forcing terms of a simulation step, broadcast vectors,
               transposed views, integer index arithmetic
  reduce       sums and extrema of a stored (batched) matrix over any axes
  reduce_expr  the same over an expression that is never stored: deviations
               from a mean, weighted sums, distances
  spmv         sparse matrix times vector(s): grid stencils and ragged rows,
               CSR, ELLPACK and 3x3 block storage, one or several vectors
  cg           Jacobi-preconditioned CG on a Poisson matrix, one or several
               right-hand sides
  cg_batched   thousands of small uneven systems solved in one launch
  cg_mixed     FP32 / BF16 inner CG inside FP64 refinement
  adjoint      a CG solve inside torch autograd, forward and backward
"""
import functools
import math

import numpy as np
import torch

import cumat_amd as cm
from cumat_amd import capi
from cumat_amd.problems import grid_laplacian
from cumat_amd.solvers import pcg_batched, pcg_ir
from cumat_amd.torch_cg import EdgeLaplacian, cg_solve

DEV = "cuda"
TORCH = {"f32": torch.float32, "f64": torch.float64, "i32": torch.int32}
NUMPY = {"f32": np.float32, "f64": np.float64, "i32": np.int32}
SIZE = {"f32": 4, "f64": 8, "i32": 4}
ROW, COL, BATCH = capi.AXIS_ROW, capi.AXIS_COL, capi.AXIS_BATCH
AXES = {"row": ROW, "col": COL, "batch": BATCH, "row+col": ROW | COL, "row+batch": ROW | BATCH,
        "col+batch": COL | BATCH, "all": capi.AXIS_ALL}
STENCILS = {"grid5": (2, 5), "grid7": (3, 7), "grid27": (3, 27)}


def listed():
    return [
        # the update of a small simulation's state: the call itself is what costs
        dict(name="cwise_axpy_small", kind="cwise", expr="axpy", dtype="f32", rows=1000, cols=3, batches=1),
        # a long vector expression: four streams in, one out
        dict(name="cwise_product_large", kind="cwise", expr="product", dtype="f32", rows=1 << 25, cols=1, batches=1),
        # symmetric part of a stack of matrices, sizes that divide by nothing
        dict(name="cwise_symmetric", kind="cwise", expr="symmetric", dtype="f32", rows=1021, cols=1021, batches=61),
        # row, column and batch sums of a stack of matrices
        dict(name="reduce_axes", kind="reduce", op="sum", axes="row,col,batch", dtype="f32", layout="col", rows=1024,
             cols=1024, batches=64),
        # squared deviation of every row from its mean, as in a normalisation
        dict(name="reduce_deviation", kind="reduce_expr", expr="deviation", axis="col", dtype="f32", rows=3000, cols=5000,
             batches=3),
        # the product of a 2D simulation
        dict(name="spmv_grid5", kind="spmv", format="csr", pattern="grid5", nx=2048, ny=2048, nz=1, dtype="f32", rhs=1),
        # a 3D finite-element matrix in double precision, one vector per displacement component
        dict(name="spmv_grid27_f64x3", kind="spmv", format="csr", pattern="grid27", nx=83, ny=71, nz=97, dtype="f64", rhs=3),
        # one small pressure solve: bound by the launches of its iterations
        dict(name="cg_128", kind="cg", pattern="grid5", nx=128, ny=128, nz=1, dtype="f32", rhs=1, tol=1e-6),
        # several right-hand sides of one matrix
        dict(name="cg_512_rhs8", kind="cg", pattern="grid5", nx=512, ny=512, nz=1, dtype="f32", rhs=8, tol=1e-6),
        # thousands of uneven systems at once
        dict(name="cg_batched", kind="cg_batched", systems=4096, low=16, high=96, tol=1e-6),
        # a large 3D solve to full FP64 accuracy
        dict(name="cg_mixed_160", kind="cg_mixed", storage="f32", nx=160, ny=160, nz=160, inner_tol=1e-5),
        # a learned coefficient field: forward and adjoint solve, gradient of every edge
        dict(name="adjoint_256x16", kind="adjoint", nx=256, ny=256, batches=16, tol=1e-7),
    ]


def _log(rng, low, high):
    """A whole number, even over its logarithm."""
    return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))


def draw(rng):
    kind = rng.choice(["cwise", "cwise", "reduce", "reduce", "reduce_expr", "reduce_expr", "spmv", "spmv", "cg",
                       "cg_batched", "cg_mixed", "adjoint"])
    if kind == "cwise":
        expr = rng.choice(["axpy", "product", "affine", "symmetric", "modulo"])
        dtype = "i32" if expr == "modulo" else rng.choice(["f32", "f32", "f64"])
        batches = _log(rng, 1, 64)
        total = _log(rng, 1000, (1 << 25) if dtype == "f64" else (1 << 26))
        rows = min(_log(rng, 1, 4096) if expr != "symmetric" else 4096, max(1, total // batches))
        cols = max(1, total // (rows * batches))
        if expr == "symmetric":
            rows = cols = max(2, int(math.sqrt(total / batches)))
        return dict(kind=kind, expr=expr, dtype=dtype, rows=rows, cols=cols, batches=batches)
    if kind in ("reduce", "reduce_expr"):
        dtype = rng.choice(["f32", "f32", "f64", "i32"] if kind == "reduce" else ["f32", "f32", "f64"])
        total = _log(rng, 2000, 1 << 26) // (2 if dtype == "f64" else 1)
        batches = _log(rng, 1, 64)
        rows = min(_log(rng, 8, 4096), max(1, total // batches))
        cols = max(1, total // (rows * batches))
        axis = rng.choice(sorted(AXES))
        if kind == "reduce":
            return dict(kind=kind, op=rng.choice(["sum", "sum", "min", "max"]), axes=axis, dtype=dtype,
                        layout=rng.choice(["col", "col", "row"]), rows=rows, cols=cols, batches=batches)
        return dict(kind=kind, expr=rng.choice(["deviation", "weighted", "distance"]), axis=axis, dtype=dtype, rows=rows,
                    cols=cols, batches=batches)
    if kind == "spmv":
        fmt = rng.choice(["csr", "csr", "csr", "ell", "block"])
        pattern = rng.choice(["grid5", "grid7", "grid27"] + (["ragged", "ragged"] if fmt == "csr" else []))
        dtype = "f32" if fmt == "block" else rng.choice(["f32", "f32", "f64"])
        rhs = rng.choice([1, 1, 2, 3, 4, 8])
        per = {"grid5": 5, "grid7": 7, "grid27": 27, "ragged": 20}[pattern] * (9 if fmt == "block" else 1)
        n = max(64, _log(rng, 20_000, 20_000_000) // per)
        if pattern == "ragged":
            return dict(kind=kind, format=fmt, pattern=pattern, nx=n, ny=1, nz=1, dtype=dtype, rhs=rhs)
        d = STENCILS[pattern][0]
        side = n ** (1.0 / d)
        nx = max(4, int(side * rng.uniform(0.7, 1.4)))
        ny = max(4, int(side * rng.uniform(0.7, 1.4)))
        return dict(kind=kind, format=fmt, pattern=pattern, nx=nx, ny=ny, nz=max(4, n // (nx * ny)) if d == 3 else 1,
                    dtype=dtype, rhs=rhs)
    if kind == "cg":
        pattern = rng.choice(["grid5", "grid5", "grid7"])
        rhs = rng.choice([1, 1, 2, 4, 8])
        n = _log(rng, 256, 1_000_000 // rhs)
        side = n ** (0.5 if pattern == "grid5" else 1 / 3)
        nx, ny = max(4, int(side * rng.uniform(0.8, 1.2))), max(4, int(side))
        return dict(kind=kind, pattern=pattern, nx=nx, ny=ny, nz=max(4, n // (nx * ny)) if pattern == "grid7" else 1,
                    dtype=rng.choice(["f32", "f32", "f64"]), rhs=rhs, tol=rng.choice([1e-4, 1e-5, 1e-6]))
    if kind == "cg_batched":
        low = rng.randint(8, 40)
        return dict(kind=kind, systems=_log(rng, 100, 4096), low=low, high=rng.randint(low, 96),
                    tol=rng.choice([1e-5, 1e-6]))
    if kind == "cg_mixed":
        s = _log(rng, 32, 144)
        return dict(kind=kind, storage=rng.choice(["f32", "bf16"]), nx=s, ny=s + rng.randint(0, 9), nz=s + rng.randint(0, 9),
                    inner_tol=rng.choice([1e-4, 1e-3]))
    return dict(kind=kind, nx=rng.randint(32, 200), ny=rng.randint(32, 200), batches=_log(rng, 1, 16),
                tol=rng.choice([1e-6, 1e-7]))


# ------------------------------------------------------------------ inputs

def _gen(seed):
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _normal(g, *shape, dtype="f32"):
    return torch.randn(*shape, generator=g, device=DEV, dtype=TORCH[dtype])


def _uniform(g, *shape, dtype="f32", low=0.0, high=1.0):
    return torch.rand(*shape, generator=g, device=DEV, dtype=TORCH[dtype]) * (high - low) + low


def _array(t, rows, cols=1, batches=1, row_major=False):
    """A torch tensor's memory as the framework's array (column-major: the
    tensor has shape (batches, cols, rows))."""
    dtype = np.uint16 if t.dtype == torch.bfloat16 else torch.empty(0, dtype=t.dtype).numpy().dtype
    return cm.DeviceArray(rows, cols, batches, dtype=dtype, row_major=row_major, ptr=t.data_ptr(), owner=t)


@functools.lru_cache(maxsize=4)
def _pattern(kind, nx, ny, nz):
    """(JA, IA) on the host. Grids: rows in C order, all neighbours of the
    stencil inside the grid, ascending columns. Ragged: 1 to 39 entries a row
    spread around the diagonal, a fixed pattern for a size."""
    if kind == "ragged":
        rng = np.random.default_rng(nx)
        per = rng.integers(1, 40, nx)
        rows = np.repeat(np.arange(nx), per)
        reach = max(1, min(nx // 2, 3000))
        cols = np.clip(rows + (rng.standard_normal(rows.size) * reach / 3).astype(np.int64), 0, nx - 1)
        key = np.unique(rows.astype(np.int64) * nx + cols)
        rows, cols = key // nx, key % nx
        JA = np.zeros(nx + 1, np.int64)
        JA[1:] = np.cumsum(np.bincount(rows, minlength=nx))
        return JA.astype(np.int32), cols.astype(np.int32)
    at = torch.arange(nx * ny * nz, device=DEV).reshape(nx, ny, nz)
    x, y, z = torch.meshgrid(*(torch.arange(k, device=DEV) for k in (nx, ny, nz)), indexing="ij")
    cols, inside = [], []
    span = (-1, 0, 1)
    for dx in span:
        for dy in span:
            for dz in span if nz > 1 else (0,):
                if kind != "grid27" and abs(dx) + abs(dy) + abs(dz) > 1:
                    continue
                inside.append(((x + dx >= 0) & (x + dx < nx) & (y + dy >= 0) & (y + dy < ny) & (z + dz >= 0)
                               & (z + dz < nz)).reshape(-1))
                cols.append((at + (dx * ny + dy) * nz + dz).reshape(-1))
    cols, inside = torch.stack(cols, 1), torch.stack(inside, 1)
    JA = torch.zeros(nx * ny * nz + 1, dtype=torch.int64, device=DEV)
    JA[1:] = torch.cumsum(inside.sum(1), 0)
    return JA.to(torch.int32).cpu().numpy(), cols[inside].to(torch.int32).cpu().numpy()


def _rows_of(JA):
    JA = torch.as_tensor(JA, device=DEV).long()
    return torch.repeat_interleave(torch.arange(JA.numel() - 1, device=DEV), JA[1:] - JA[:-1])


def _vectors(case, g):
    """What each family's inputs are, as torch tensors, in the case's type."""
    kind = case["kind"]
    if kind == "cwise":
        R, C, B, dt, e = case["rows"], case["cols"], case["batches"], case["dtype"], case["expr"]
        if e == "modulo":
            draw_int = functools.partial(torch.randint, generator=g, device=DEV, dtype=torch.int32)
            return {"a": draw_int(0, 1 << 30, (B, C, R)), "b": draw_int(1, 1 << 12, (B, C, R))}
        if e == "affine":
            return {"a": _normal(g, B, C, R, dtype=dt), "u": _normal(g, 1, 1, R, dtype=dt), "v": _normal(g, 1, C, 1, dtype=dt)}
        return {k: _normal(g, B, C, R, dtype=dt) for k in {"axpy": "ab", "product": "abcd", "symmetric": "a"}[e]}
    R, C, B, dt = case["rows"], case["cols"], case["batches"], case["dtype"]
    shape = (B, R, C) if case.get("layout") == "row" else (B, C, R)
    if dt == "i32":
        return {"a": torch.randint(-1000, 1001, shape, generator=g, device=DEV, dtype=torch.int32)}
    # positive values: a sum is then as large as its terms, and its error means something
    out = {"a": _uniform(g, *shape, dtype=dt)}
    if kind == "reduce_expr":
        axis = AXES[case["axis"]]
        if case["expr"] == "distance":
            out["b"] = _uniform(g, *shape, dtype=dt)
        elif case["expr"] == "weighted":  # a weight for every position along the reduced axes
            out["b"] = _uniform(g, B if axis & BATCH else 1, C if axis & COL else 1, R if axis & ROW else 1, dtype=dt)
        else:  # the mean over the reduced axes
            out["b"] = out["a"].mean(dim=[d for d, bit in ((0, BATCH), (1, COL), (2, ROW)) if axis & bit], keepdim=True)
    return out


def _matrix_values(case, g, JA, IA):
    """Stored values of an M-matrix: off-diagonals in [-1, -0.1], a diagonal that dominates."""
    rows = _rows_of(JA)
    cols = torch.as_tensor(IA, device=DEV).long()
    v = -_uniform(g, cols.numel(), dtype="f64", low=0.1, high=1.0)
    v = torch.where(rows == cols, 30.0, v)
    return v, rows, cols


def _batched_systems(case, g):
    """One block-diagonal CSR matrix of uneven shifted 2D Poisson systems. A
    case's sides are the same for every seed; shifts and right-hand sides are not."""
    S = case["systems"]
    side = torch.randint(case["low"], case["high"] + 1, (S,), generator=_gen(S), device=DEV)
    shift = _uniform(g, S)
    n = side * side
    off = torch.zeros(S + 1, dtype=torch.int64, device=DEV)
    off[1:] = torch.cumsum(n, 0)
    total = int(off[-1])
    which = torch.repeat_interleave(torch.arange(S, device=DEV), n)
    row = torch.arange(total, device=DEV)
    w = side[which]
    local = row - off[which]
    x, y = local // w, local % w
    inside = torch.stack([x > 0, y > 0, torch.ones_like(x, dtype=torch.bool), y < w - 1, x < w - 1], 1)
    cols = torch.stack([row - w, row - 1, row, row + 1, row + w], 1)
    vals = torch.full((total, 5), -1.0, device=DEV)
    vals[:, 2] = 4.0 + shift[which]
    JA = torch.zeros(total + 1, dtype=torch.int64, device=DEV)
    JA[1:] = torch.cumsum(inside.sum(1), 0)
    return {"JA": JA.int(), "IA": cols[inside].int(), "vals": vals[inside], "off": off.int(), "side": side,
            "diag": 4.0 + shift, "b": _uniform(g, total, low=-1.0)}


def _edge_fields(case, g):
    """Log-normal coefficients of every edge of a 3D grid, boundary edges included (FP64)."""
    nx, ny, nz = case["nx"], case["ny"], case["nz"]
    return [torch.exp(_normal(g, *s, dtype="f64")) for s in ((nx + 1, ny, nz), (nx, ny + 1, nz), (nx, ny, nz + 1))]


def _grid_operator(fields):
    """v -> A v for the edge Laplacian of these coefficients; v: (..., *grid)."""
    d = len(fields)
    low = [f.narrow(f.dim() - d + a, 0, f.shape[f.dim() - d + a] - 1) for a, f in enumerate(fields)]
    high = [f.narrow(f.dim() - d + a, 1, f.shape[f.dim() - d + a] - 1) for a, f in enumerate(fields)]
    diag = sum(low) + sum(high)

    def apply(v):
        out = diag * v
        for a in range(d):
            k = v.dim() - d + a
            m = v.shape[k] - 1
            f = low[a].narrow(low[a].dim() - d + a, 1, m)
            out.narrow(k, 1, m).sub_(f * v.narrow(k, 0, m))
            out.narrow(k, 0, m).sub_(f * v.narrow(k, 1, m))
        return out

    return apply, diag


def _theta_fields(theta, nx, ny):
    """The edge vector of a 2D grid (x edges, then y edges) as fields."""
    split = (nx + 1) * ny
    return [theta[:, :split].reshape(-1, nx + 1, ny), theta[:, split:].reshape(-1, nx, ny + 1)]


@functools.lru_cache(maxsize=2)
def _edge_laplacian(nx, ny):
    return EdgeLaplacian(grid_laplacian((nx, ny), lambda shape: np.ones(shape)), device=DEV)


# ------------------------------------------------------------------- cases

def prepare(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind == "cwise":
        R, C, B, e = case["rows"], case["cols"], case["batches"], case["expr"]
        t = _vectors(case, g)
        out = torch.empty(B, C, R, dtype=TORCH[case["dtype"]], device=DEV)
        arr = {k: _array(v, v.shape[2], v.shape[1], v.shape[0]) for k, v in t.items()}
        return {"kind": kind, "expr": e, "arr": arr, "out": out, "dst": _array(out, R, C, B)}
    if kind in ("reduce", "reduce_expr"):
        R, C, B = case["rows"], case["cols"], case["batches"]
        t = _vectors(case, g)
        row_major = case.get("layout") == "row"
        arr = {k: _array(v, *((v.shape[1], v.shape[2]) if row_major else (v.shape[2], v.shape[1])), v.shape[0],
                         row_major=row_major) for k, v in t.items()}
        todo = []
        for name in case["axes"].split(",") if kind == "reduce" else [case["axis"]]:
            ax = AXES[name]
            o = (1 if ax & ROW else R, 1 if ax & COL else C, 1 if ax & BATCH else B)
            out = torch.empty((o[2], o[0], o[1]) if row_major else (o[2], o[1], o[0]), dtype=TORCH[case["dtype"]],
                              device=DEV)
            todo.append((ax, out, _array(out, *o, row_major=row_major)))
        return {"kind": kind, "op": case.get("op", "sum"), "expr": case.get("expr"), "arr": arr, "todo": todo}
    if kind == "spmv":
        JA, IA = _pattern(case["pattern"], case["nx"], case["ny"], case["nz"])
        n, B, dt, fmt = JA.size - 1, case["rhs"], case["dtype"], case["format"]
        v, rows, cols = _matrix_values(case, g, JA, IA)
        entry = 4 if fmt == "block" else 1  # floats of a vector entry
        x = _normal(g, B, n * entry, dtype=dt)
        y = torch.empty_like(x)
        if fmt == "csr":
            A = cm.SparseMatrix(cm.SparsityPattern(n, n, JA, IA), _array(v.to(TORCH[dt]), IA.size))
        elif fmt == "ell":
            width = int(np.diff(JA).max())
            slot = torch.arange(IA.size, device=DEV) - torch.as_tensor(JA, device=DEV).long()[rows]
            idx = torch.full((n, width), -1, dtype=torch.int32, device=DEV)
            val = torch.zeros(n, width, dtype=TORCH[dt], device=DEV)
            idx[rows, slot], val[rows, slot] = cols.int(), v.to(TORCH[dt])
            A = cm.ELLMatrix(n, n, idx.cpu().numpy(), val.cpu().numpy())
        else:
            A = cm.BlockSparseMatrix(cm.SparsityPattern(n, n, JA, IA), 3, _blocks(v, g).float().cpu().numpy())
        return {"kind": kind, "A": A, "x": _array(x, n * entry, 1, B), "y": _array(y, n * entry, 1, B), "out": y}
    if kind == "cg":
        JA, IA = _pattern(case["pattern"], case["nx"], case["ny"], case["nz"])
        n, B, dt = JA.size - 1, case["rhs"], case["dtype"]
        v = np.where(IA == np.repeat(np.arange(n), np.diff(JA)), STENCILS[case["pattern"]][1] - 1.0, -1.0)
        A = cm.SparseMatrix.from_csr(n, n, JA, IA, v.astype(NUMPY[dt]))
        b = _uniform(g, B, n, dtype=dt, low=-1.0)
        x = torch.empty_like(b)
        solver = cm.ConjugateGradient(A).setTolerance(case["tol"]).setMaxIterations(20000)
        return {"kind": kind, "solver": solver, "b": _array(b, n, 1, B), "x": _array(x, n, 1, B), "out": x}
    if kind == "cg_batched":
        s = _batched_systems(case, g)
        S, n = case["systems"], s["b"].numel()
        x = torch.empty_like(s["b"])
        its, errs = torch.empty(S, dtype=torch.int32, device=DEV), torch.empty(S, device=DEV)
        arr = {k: _array(s[k], s[k].numel()) for k in ("off", "JA", "IA", "vals", "b")}
        return {"kind": kind, "arr": arr, "tol": case["tol"], "x": _array(x, n), "its": _array(its, S),
                "errs": _array(errs, S), "out": x}
    if kind == "cg_mixed":
        JA, IA = _pattern("grid7", case["nx"], case["ny"], case["nz"])
        n = JA.size - 1
        vals = _edge_values(_edge_fields(case, g), JA, IA)
        b = _uniform(g, n, dtype="f64", low=-1.0)
        x = torch.empty_like(b)
        return {"kind": kind, "JA": cm.DeviceArray.from_numpy(JA), "IA": cm.DeviceArray.from_numpy(IA),
                "vals": _array(vals, IA.size), "b": _array(b, n), "x": _array(x, n), "out": x,
                "storage": case["storage"], "inner_tol": case["inner_tol"]}
    lap = _edge_laplacian(case["nx"], case["ny"])
    theta, b, target = _adjoint_inputs(case, g, lap.n, lap.nedges)
    return {"kind": kind, "lap": lap, "theta": theta.requires_grad_(), "b": b.requires_grad_(), "target": target,
            "tol": case["tol"]}


def _blocks(v, g):
    """3x3 blocks of the stored scalars: v * (I + a small coupling), rows padded to four floats."""
    k = 0.1 * _normal(g, v.numel(), 3, 3, dtype="f64")
    k += torch.eye(3, device=DEV, dtype=torch.float64)
    out = torch.zeros(v.numel(), 3, 4, device=DEV, dtype=torch.float64)
    out[:, :, :3] = v[:, None, None] * k
    return out


def _edge_values(fields, JA, IA):
    """CSR values of the edge Laplacian on the 7-point pattern (C order, ascending columns)."""
    nx, ny, nz = fields[1].shape[0], fields[0].shape[1], fields[0].shape[2]
    low = [f.narrow(a, 0, f.shape[a] - 1) for a, f in enumerate(fields)]
    high = [f.narrow(a, 1, f.shape[a] - 1) for a, f in enumerate(fields)]
    slots = [-low[0], -low[1], -low[2], sum(low) + sum(high), -high[2], -high[1], -high[0]]
    at = [torch.arange(k, device=DEV).reshape([-1 if a == b else 1 for b in range(3)]) for a, k in enumerate((nx, ny, nz))]
    inside = [at[0] > 0, at[1] > 0, at[2] > 0, at[0] >= 0, at[2] < nz - 1, at[1] < ny - 1, at[0] < nx - 1]
    inside = torch.stack([m.expand(nx, ny, nz).reshape(-1) for m in inside], 1)
    return torch.stack([s.reshape(-1) for s in slots], 1)[inside]


def _adjoint_inputs(case, g, n, nedges):
    B = case["batches"]
    return torch.exp(0.5 * _normal(g, B, nedges)), _uniform(g, B, n, low=-1.0), _normal(g, B, n)


def run(state):
    kind = state["kind"]
    if kind == "cwise":
        arr, e = state["arr"], state["expr"]
        if e == "axpy":
            ex = arr["a"].expr() * 0.75 + arr["b"]
        elif e == "product":
            ex = (arr["a"].expr() + arr["b"]) * (arr["c"].expr() - arr["d"])
        elif e == "affine":
            ex = arr["a"].expr() * arr["u"] + arr["v"]
        elif e == "symmetric":
            a = arr["a"].expr()
            ex = (a + a.T) * 0.5
        else:
            ex = arr["a"].expr() % arr["b"]
        cm.assign(state["dst"], ex)
        return state["out"]
    if kind == "reduce":
        for axis, _, dst in state["todo"]:
            cm.reduce(state["arr"]["a"], state["op"], axis, out=dst)
        return [out for _, out, _ in state["todo"]]
    if kind == "reduce_expr":
        a, b = state["arr"]["a"].expr(), state["arr"]["b"]
        axis, out, dst = state["todo"][0]
        cm.reduce(a * b if state["expr"] == "weighted" else (a - b).cwiseAbs2(), "sum", axis, out=dst)
        return out
    if kind == "spmv":
        state["A"].matvec(state["x"], out=state["y"])
        return state["out"]
    if kind == "cg":
        state["solver"].solve(state["b"], x=state["x"])
        return state["out"]
    if kind == "cg_batched":
        a = state["arr"]
        pcg_batched(a["off"], a["JA"], a["IA"], a["vals"], a["b"], state["x"], state["tol"], 2000, state["its"], state["errs"])
        return state["out"]
    if kind == "cg_mixed":
        pcg_ir(state["JA"], state["IA"], state["vals"], state["b"], state["x"], storage=state["storage"], tol=1e-12,
               inner_tol=state["inner_tol"])
        return state["out"]
    theta, b = state["theta"], state["b"]
    x = cg_solve(theta, b, state["lap"], tol=state["tol"])
    gtheta, gb = torch.autograd.grad(x, (theta, b), x.detach() - state["target"])  # loss 0.5 |x - target|^2
    return x.detach(), gtheta, gb


# ---------------------------------------------------------- what it has to do

def _entries(case):
    """(rows, stored entries) of a case's matrix, counted without building a grid's."""
    nx, ny, nz = case["nx"], case["ny"], case.get("nz", 1)
    n, pattern = nx * ny * nz, case.get("pattern", "grid7" if case["kind"] == "cg_mixed" else "grid5")
    if pattern == "ragged":
        return n, int(_pattern(pattern, nx, ny, nz)[0][-1])
    if pattern == "grid27":
        return n, (3 * nx - 2) * (3 * ny - 2) * (3 * nz - 2)
    nnz = n + 2 * ((nx - 1) * ny * nz + nx * (ny - 1) * nz) + (2 * nx * ny * (nz - 1) if pattern == "grid7" else 0)
    return n, nnz


def _iterations(case):
    """About how many CG iterations a grid needs: they grow with its side and the digits asked for."""
    digits = -math.log10(case["tol"]) / 6.0
    side = max(case["nx"], case["ny"], case.get("nz", 1))
    return max(4.0, {"cg": 2.5 if case.get("nz", 1) == 1 else 1.7, "adjoint": 3.3}[case["kind"]] * side * digits)


def work(case):
    kind = case["kind"]
    if kind in ("cwise", "reduce", "reduce_expr"):
        R, C, B, s = case["rows"], case["cols"], case["batches"], SIZE[case["dtype"]]
        n = R * C * B
        if kind == "cwise":
            reads = {"axpy": 2 * n, "product": 4 * n, "affine": n + R + C, "symmetric": n, "modulo": 2 * n}[case["expr"]]
            return {"bytes": s * (reads + n), "flops": {"product": 3, "modulo": 1}.get(case["expr"], 2) * n}
        out = 0
        names = case["axes"].split(",") if kind == "reduce" else [case["axis"]]
        for name in names:
            ax = AXES[name]
            out += (1 if ax & ROW else R) * (1 if ax & COL else C) * (1 if ax & BATCH else B)
        reads = n * (2 if case.get("expr") == "distance" else 1)
        # each of several reductions is a call of its own and reads the array again
        return {"bytes": s * (reads * len(names) + out), "flops": n * len(names) * (3 if kind == "reduce_expr" else 1)}
    if kind == "spmv":
        n, nnz = _entries(case)
        B, s = case["rhs"], SIZE[case["dtype"]]
        if case["format"] == "block":
            return {"bytes": nnz * (48 + 4) + 4 * n + 32 * n * B, "flops": 2 * 9 * nnz * B}
        return {"bytes": nnz * (4 + s) + 4 * n + 2 * s * n * B, "flops": 2 * nnz * B}
    if kind in ("cg", "adjoint"):
        # an iteration reads the matrix and nine vectors' worth of reads and writes (product, two updates, two sums)
        n, nnz = _entries(case)
        s = SIZE[case.get("dtype", "f32")]
        B = case.get("rhs", case.get("batches"))
        matrix = nnz * (4 + s * (B if kind == "adjoint" else 1)) + 4 * n
        its = _iterations(case) * (2 if kind == "adjoint" else 1)
        return {"bytes": its * (matrix + 9 * s * n * B), "flops": its * B * (2 * nnz + 12 * n)}
    if kind == "cg_batched":
        # 22 bytes per stored entry and row of a matrix that is read once; its iterations stay on the chip
        side = (case["low"] + case["high"]) / 2.0
        n = case["systems"] * (side * side + (case["high"] - case["low"]) ** 2 / 12.0)
        return {"bytes": n * (5 * 8 + 4 + 8), "flops": n * 22 * 60}
    n, nnz = _entries(case)
    its = 8.7 * max(case["nx"], case["ny"], case["nz"])
    value = 4 if case["storage"] == "f32" else 2
    return {"bytes": its * (nnz * (4 + value) + 40 * n) + 4 * (12 * nnz + 24 * n), "flops": its * (2 * nnz + 12 * n)}


def tolerance(case):
    kind = case["kind"]
    if case.get("dtype") == "i32":
        return "exact"
    double = case.get("dtype") == "f64"
    if kind == "cwise":
        return {"rel": 4e-16 if double else 2e-7}
    if kind in ("reduce", "reduce_expr"):
        if case.get("op") in ("min", "max"):
            return "exact"
        return {"rel": 4e-15 if double else 2e-6}
    if kind == "spmv":
        return {"rel": 1e-15 if double else 3e-7}
    if kind == "cg":  # stops at a residual: the answer is off by up to that, times the condition
        return {"rel": 12 * case["tol"]}
    if kind == "cg_batched":
        return {"rel": 10 * case["tol"]}
    if kind == "cg_mixed":
        return {"rel": 2e-11}
    return {"rel": 3e-4}  # the gradient of the coefficients; x and lambda are ten times closer


# ------------------------------------------------------------------ in 64 bits

def _solve64(apply, diag, b, tol, dims):
    """Jacobi CG in FP64 on tensors; every leading index is a system of its own. dims: the grid axes of b."""
    x, r = torch.zeros_like(b), b.clone()
    z = r / diag
    p = z.clone()
    rz = (r * z).sum(dims, keepdim=True)
    stop = tol * tol * (b * b).sum(dims, keepdim=True)
    for it in range(20000):
        q = apply(p)
        alpha = rz / (p * q).sum(dims, keepdim=True).clamp_min(1e-300)
        x += alpha * p
        r -= alpha * q
        if it % 16 == 15 and bool(((r * r).sum(dims, keepdim=True) <= stop).all()):
            break
        z = r / diag
        new = (r * z).sum(dims, keepdim=True)
        p = z + (new / rz.clamp_min(1e-300)) * p
        rz = new
    return x


def exact(case, seed):
    kind, g = case["kind"], _gen(seed)
    if kind in ("cwise", "reduce", "reduce_expr"):
        t = {k: (v.long() if v.dtype == torch.int32 else v.double()) for k, v in _vectors(case, g).items()}
        a = t["a"]
        if kind == "cwise":
            e = case["expr"]
            if e == "axpy":
                return a * 0.75 + t["b"]
            if e == "product":
                return (a + t["b"]) * (t["c"] - t["d"])
            if e == "affine":
                return a * t["u"] + t["v"]
            return (a + a.transpose(1, 2)) * 0.5 if e == "symmetric" else (a % t["b"]).int()
        if kind == "reduce_expr":
            a = a * t["b"] if case["expr"] == "weighted" else (a - t["b"]).square()
        row_major = case.get("layout") == "row"
        outs = []
        for name in case["axes"].split(",") if kind == "reduce" else [case["axis"]]:
            ax = AXES[name]
            dims = [d for d, bit in ((0, BATCH), (2, COL if row_major else ROW), (1, ROW if row_major else COL)) if ax & bit]
            op = case.get("op", "sum")
            o = a.sum(dims, keepdim=True) if op == "sum" else getattr(torch, "a" + op)(a, dims, keepdim=True)
            outs.append(o.int() if case["dtype"] == "i32" else o)
        return outs if kind == "reduce" else outs[0]
    if kind == "spmv":
        JA, IA = _pattern(case["pattern"], case["nx"], case["ny"], case["nz"])
        n, B, dt = JA.size - 1, case["rhs"], case["dtype"]
        v, rows, cols = _matrix_values(case, g, JA, IA)
        if case["format"] == "block":
            x = _normal(g, B, n * 4, dtype=dt).double().reshape(B, n, 4)
            v = _blocks(v, g).float().double()
            out = torch.zeros(B, n, 4, dtype=torch.float64, device=DEV)
            for k in range(B):
                out[k, :, :3].index_add_(0, rows, (v * x[k][cols][:, None, :]).sum(2))
            return out.reshape(B, n * 4)
        v = v.to(TORCH[dt]).double()
        x = _normal(g, B, n, dtype=dt).double()
        out = torch.zeros_like(x)
        for k in range(B):
            out[k].index_add_(0, rows, v * x[k][cols])
        return out
    if kind == "cg":
        shape = [k for k in (case["nx"], case["ny"], case["nz"]) if k > 1]
        d = len(shape)
        b = _uniform(g, case["rhs"], math.prod(shape), dtype=case["dtype"], low=-1.0).double().reshape(-1, *shape)
        fields = [torch.ones([k + (a == c) for c, k in enumerate(shape)], dtype=torch.float64, device=DEV) for a in range(d)]
        apply, diag = _grid_operator(fields)
        return _solve64(apply, diag, b, 1e-12, list(range(1, d + 1))).reshape(case["rhs"], -1)
    if kind == "cg_batched":  # every system in the corner of a grid of the largest side
        s = _batched_systems(case, g)
        H, S = case["high"], case["systems"]
        side, k = s["side"][:, None, None], torch.arange(H, device=DEV)
        mask = (k[None, :, None] < side) & (k[None, None, :] < side)
        b = torch.zeros(S, H, H, dtype=torch.float64, device=DEV)
        b[mask] = s["b"].double()
        diag = s["diag"].double()[:, None, None]

        def apply(v):
            out = diag * v
            for a in (1, 2):
                out.narrow(a, 1, H - 1).sub_(v.narrow(a, 0, H - 1))
                out.narrow(a, 0, H - 1).sub_(v.narrow(a, 1, H - 1))
            return out * mask

        return _solve64(apply, diag, b, 1e-12, [1, 2])[mask]
    if kind == "cg_mixed":
        apply, diag = _grid_operator(_edge_fields(case, g))
        b = _uniform(g, case["nx"] * case["ny"] * case["nz"], dtype="f64", low=-1.0)
        return _solve64(apply, diag, b.reshape(diag.shape), 1e-14, [0, 1, 2]).reshape(-1)
    nx, ny = case["nx"], case["ny"]
    theta, b, target = (t.double() for t in _adjoint_inputs(case, g, nx * ny, (nx + 1) * ny + nx * (ny + 1)))
    fields = _theta_fields(theta, nx, ny)
    apply, diag = _grid_operator(fields)
    x = _solve64(apply, diag, b.reshape(-1, nx, ny), 1e-12, [1, 2])
    lam = _solve64(apply, diag, x - target.reshape(-1, nx, ny), 1e-12, [1, 2])
    grads = []
    for axis in (1, 2):  # dL/dtheta_e = -(lam_i - lam_j)(x_i - x_j), zero outside the grid
        pad = [0, 0, 1, 1] if axis == 1 else [1, 1, 0, 0]
        dx, dl = (torch.nn.functional.pad(v, pad).diff(dim=axis) for v in (x, lam))
        grads.append(-(dx * dl).reshape(len(dx), -1))
    return x.reshape(len(x), -1), torch.cat(grads, 1), lam.reshape(len(lam), -1)
