"""The CG iteration over a matrix laid out by diagonals (cg_dia.hpp): the
forms it takes (tile edges, missing entries, several right-hand sides, values
per batch, FP64) and those it must leave to the CSR product (too many
diagonals, columns out of order, an entry that the sample did not show),
against the CPU oracle; and which solves lay their matrix out at all."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def banded(n, offsets, seed, drop=0.0, dtype=np.float32):
    """A symmetric positive definite matrix whose entries lie at +-offsets;
    'drop' of the off-diagonal pairs are not stored."""
    rng = np.random.default_rng(seed)
    rows, cols, vals = [np.arange(n)], [np.arange(n)], [np.zeros(n)]
    diag = np.full(n, 2e-3)
    for o in offsets:
        i = np.arange(n - o)
        i = i[rng.uniform(size=i.size) >= drop]
        v = -rng.uniform(0.5, 1.0, i.size)
        rows += [i, i + o]
        cols += [i + o, i]
        vals += [v, v]
        np.add.at(diag, i, -v)
        np.add.at(diag, i + o, -v)
    vals[0] = diag
    rows, cols, vals = map(np.concatenate, (rows, cols, vals))
    order = np.lexsort((cols, rows))
    JA = np.zeros(n + 1, np.int32)
    JA[1:] = np.cumsum(np.bincount(rows, minlength=n))
    return JA, cols[order].astype(np.int32), vals[order].astype(dtype)


def check(cm, orc, JA, IA, V, rhs=1, dtype=np.float32, tol=1e-5, path=1, diagonals=None):
    """diagonals: whether the solve has to run over them."""
    n = JA.size - 1
    b = np.random.default_rng(n).uniform(-1, 1, n * rhs).astype(dtype)
    cg = cm.ConjugateGradient(cm.SparseMatrix.from_csr(n, n, JA, IA, V), path=path)
    cg.setTolerance(tol).setMaxIterations(5000)
    cm.reset_counters()
    x = cg.solve(cm.DeviceArray.from_numpy(b, rows=n, batches=rhs)).numpy().reshape(rhs, n)
    if diagonals is not None:
        assert (cm.counters()["CgDiagonals"] > 0) == diagonals
    _, it, _ = orc.pcg(JA, IA, V, b, n, batches=rhs, tol=tol, max_iter=5000)
    assert cg.error() <= tol
    # FP32 recurrences of a system of condition ~1e3 drift apart by a few per cent of the iterations
    assert abs(cg.iterations() - it) <= (2 if dtype == np.float64 else 2 + it // 20)
    A = V.astype(np.float64)
    for k in range(rhs):
        # the true residual: the recurrence's (<= tol) and the rounding of x, n_iter updates of relative size eps
        y = np.add.reduceat(A * x[k].astype(np.float64)[IA], JA[:-1])
        bk = b.reshape(rhs, n)[k].astype(np.float64)
        scale = np.abs(A).max() * 4 * np.linalg.norm(x[k]) / np.linalg.norm(bk)
        bound = tol + cg.iterations() * np.finfo(dtype).eps * scale
        assert np.linalg.norm(bk - y) / np.linalg.norm(bk) <= bound


@pytest.mark.parametrize("n", [2047, 2048, 2049, 2559, 2560, 2561, 70001])
@pytest.mark.parametrize("offsets", [(1,), (1, 37), (1, 5, 31), (1, 2, 3, 4, 5, 11, 12, 13, 40, 41, 42, 43, 44)])
def test_diagonals(gpu, orc, n, offsets):
    check(gpu, orc, *banded(n, offsets, n), diagonals=n >= 2048)  # fewer unknowns keep the CSR product


@pytest.mark.parametrize("rhs,dtype", [(2, np.float32), (3, np.float32), (4, np.float64), (5, np.float32)])
def test_right_hand_sides(gpu, orc, rhs, dtype):
    check(gpu, orc, *banded(3001, (1, 60), rhs, drop=0.1, dtype=dtype), rhs=rhs, dtype=dtype,
          tol=1e-5 if dtype == np.float32 else 1e-10, diagonals=True)


@pytest.mark.parametrize("offsets", [(1,), (1, 37), (1, 5, 31)])
@pytest.mark.parametrize("n,rhs", [(255, 1), (256, 2), (257, 16), (1000, 17), (5001, 3), (70001, 1)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_two_launch_form(gpu, orc, offsets, n, rhs, dtype):
    """3, 5 and 7 diagonals, block edges, and both folds of the right-hand sides' sums."""
    check(gpu, orc, *banded(n, offsets, n, drop=0.1, dtype=dtype), rhs=rhs, dtype=dtype,
          tol=1e-5 if dtype == np.float32 else 1e-10, path=3, diagonals=True)


def test_two_launch_form_leaves_other_counts(gpu, orc):
    check(gpu, orc, *banded(3000, (1, 2, 3, 50), 8), path=3, diagonals=False)  # 9 diagonals
    check(gpu, orc, *banded(3000, (), 9), path=3, diagonals=False)


@pytest.mark.parametrize("path", [1, 3])
def test_iteration_limit_behind_the_switch(gpu, orc, path):
    cm = gpu
    n, limit = 4000, 103
    JA, IA, V = banded(n, (1, 61), 10, dtype=np.float64)
    b = np.random.default_rng(10).uniform(-1, 1, n)
    cg = cm.ConjugateGradient(cm.SparseMatrix.from_csr(n, n, JA, IA, V), path=path)
    cm.reset_counters()
    x = cg.setTolerance(1e-14).setMaxIterations(limit).solve(cm.DeviceArray.from_numpy(b)).numpy().reshape(-1)
    assert 0 < cm.counters()["CgDiagonals"] < limit and cg.iterations() == limit
    xo, it, _ = orc.pcg(JA, IA, V, b, n, tol=1e-14, max_iter=limit)
    assert it == limit
    # rounding grows along the recurrences, far from the residual that is left
    np.testing.assert_allclose(x, xo, rtol=0, atol=1e-8 * np.abs(xo).max())


@pytest.mark.parametrize("half", [4, 6, 12, 13, 15])
@pytest.mark.parametrize("rhs,dtype", [(1, np.float32), (2, np.float64)])
def test_several_chains(gpu, orc, half, rhs, dtype):
    """9 to 31 diagonals: four chains of a row, from 27 on eight, and remainders of each."""
    JA, IA, V = banded(6000, tuple(range(1, half)) + (700,), half, drop=0.1, dtype=dtype)
    check(gpu, orc, JA, IA, V, rhs=rhs, dtype=dtype, tol=1e-5 if dtype == np.float32 else 1e-10, diagonals=True)


def test_four_rows_per_lane(gpu, orc):
    check(gpu, orc, *banded((1 << 21) + 777, (1, 1500), 3), tol=1e-3, diagonals=True)


def test_too_many_diagonals(gpu, orc):
    check(gpu, orc, *banded(2600, tuple(range(1, 34, 2)), 4), diagonals=False)  # 35 diagonals


def test_columns_out_of_order(gpu, orc):
    JA, IA, V = banded(2500, (1, 50), 5)
    for i in range(0, 2500, 7):  # reversed rows
        s = slice(JA[i], JA[i + 1])
        IA[s], V[s] = IA[s][::-1].copy(), V[s][::-1].copy()
    check(gpu, orc, JA, IA, V, diagonals=False)


def test_entry_outside_the_sample(gpu, orc):
    n = 50001
    JA, IA, V = banded(n, (1, 200), 6)
    # one more coupling, of two rows that a sample of every 24th row does not hold
    i, j = 1001, 30007
    rows = np.repeat(np.arange(n), np.diff(JA))
    rows = np.concatenate([rows, [i, j]])
    cols = np.concatenate([IA, [j, i]])
    vals = np.concatenate([V, [-0.25, -0.25]]).astype(np.float32)
    vals[(rows == cols) & ((rows == i) | (rows == j))] += 0.25
    order = np.lexsort((cols, rows))
    JA2 = np.zeros(n + 1, np.int32)
    JA2[1:] = np.cumsum(np.bincount(rows, minlength=n))
    check(gpu, orc, JA2, cols[order].astype(np.int32), vals[order], diagonals=False)


@pytest.mark.parametrize("batches", [2, 5])
def test_values_per_batch(gpu, orc, batches):
    import torch
    from cumat_amd.problems import grid_laplacian, lognormal_sampler
    from cumat_amd.torch_cg import EdgeLaplacian
    rng = np.random.default_rng(batches)
    P = grid_laplacian((41, 37), lognormal_sampler(rng))
    lap = EdgeLaplacian(P)
    theta = torch.as_tensor(np.exp(rng.standard_normal((batches, P["nedges"]))), device="cuda")
    b = torch.as_tensor(rng.uniform(-1, 1, (batches, P["n"])), device="cuda")
    vals = lap.assemble(theta)
    gpu.reset_counters()
    x, its, errs = lap.solve(vals, b, 1e-11, 5000)
    assert gpu.counters()["CgDiagonals"] > 0 and max(errs) <= 1e-11
    for k in range(batches):
        xo, it, _ = orc.pcg(P["JA"], P["IA"], vals[k].cpu().numpy(), b[k].cpu().numpy(), P["n"], tol=1e-11,
                            max_iter=5000)
        assert abs(its[k] - it) <= 2
        np.testing.assert_allclose(x[k].cpu().numpy(), xo, rtol=0, atol=1e-8 * np.abs(xo).max())


def poisson_solver(cm, side, path):
    from cumat_amd.problems import poisson2d
    n = side * side
    JA, IA, V = poisson2d(side)
    b = cm.DeviceArray.from_numpy(np.random.default_rng(side).uniform(-1, 1, n).astype(np.float32))
    return cm.ConjugateGradient(cm.SparseMatrix.from_csr(n, n, JA, IA, V), path=path), b


def layouts(cm, cg, b, tol, max_iter=2000):
    """(iterations, layouts queued, whether iterations ran over the diagonals)"""
    cm.reset_counters()
    cg.setTolerance(tol).setMaxIterations(max_iter).solve(b)
    c = cm.counters()
    return cg.iterations(), c["CgLayout"], c["CgDiagonals"] > 0


@pytest.mark.parametrize("path,side", [(1, 128), (1, 600), (3, 128)])
def test_short_solves_lay_nothing_out(gpu, path, side):
    """Below about 30 iterations the layout costs more than it gains."""
    cm = gpu
    cg, b = poisson_solver(cm, side, path)
    seen = [layouts(cm, cg, b, tol) for tol in (0.5, 0.3, 0.2, 0.14, 0.1, 0.07, 0.05)]
    assert min(it for it, _, _ in seen) <= 8 and max(it for it, _, _ in seen) >= 20
    for it, queued, used in seen:
        if it <= 32:
            assert (queued, used) == (0, False), it
    assert layouts(cm, cg, b, 0.0, 30)[1:] == (0, False)  # too few iterations allowed
    it, queued, used = layouts(cm, cg, b, 1e-6)
    assert it > 150 and (queued, used) == (1, True)


def test_the_switch_is_reproducible(gpu):
    cm = gpu
    cg, b = poisson_solver(cm, 300, 1)
    runs = [cg.setTolerance(1e-6).setMaxIterations(2000).solve(b).numpy().tobytes() for _ in range(5)]
    assert len(set(runs)) == 1
