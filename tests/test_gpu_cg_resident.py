"""The one-workgroup CG with its matrix in registers (cg_resident_kernel):
row counts at the edges of its tiles, and the systems it has to leave to the
CSR walk (an offset beyond the guard, more diagonals than the mean row length
says, columns out of order), against the CPU oracle."""
import numpy as np
import pytest

from test_gpu_cg_dia import banded

pytestmark = pytest.mark.gpu


def solve(cm, orc, JA, IA, V, path=2, guess=None, tol=1e-5, walks=None):
    n = JA.size - 1
    dtype = V.dtype
    b = np.random.default_rng(n).uniform(-1, 1, n).astype(dtype)
    cg = cm.ConjugateGradient(cm.SparseMatrix.from_csr(n, n, JA, IA, V), path=path)
    cg.setTolerance(tol).setMaxIterations(4000)
    bd = cm.DeviceArray.from_numpy(b)
    cm.reset_counters()
    x = (cg.solve(bd) if guess is None else cg.solveWithGuess(bd, cm.DeviceArray.from_numpy(guess))).numpy()
    _, it, _ = orc.pcg(JA, IA, V, b, n, x0=guess, tol=tol, max_iter=4000)
    if walks is not None:
        assert cm.counters()["CgWalk"] == int(walks)
    assert cg.error() <= tol
    assert abs(cg.iterations() - it) <= (2 if dtype == np.float64 else 2 + it // 20)
    y = np.add.reduceat(V.astype(np.float64) * x.astype(np.float64)[IA], JA[:-1])
    b64 = b.astype(np.float64)
    # the recurrence's residual, and the rounding of one update of x per iteration
    bound = tol + (1 + cg.iterations()) * np.finfo(dtype).eps * 4 * np.abs(V).max() * np.linalg.norm(x) / np.linalg.norm(b64)
    assert np.linalg.norm(b64 - y) / np.linalg.norm(b64) <= bound
    return cg


@pytest.mark.parametrize("n", [1, 2, 63, 64, 65, 511, 512, 513, 1025, 2047, 4097, 6145, 9215, 9216])
def test_five_diagonals(gpu, orc, n):
    offsets = [o for o in (1, 96) if o < n]
    solve(gpu, orc, *banded(n, offsets, n, drop=0.05 if n > 100 else 0.0), walks=False)


@pytest.mark.parametrize("n", [513, 2048, 2049, 6143, 7000])
def test_seven_diagonals(gpu, orc, n):
    solve(gpu, orc, *banded(n, (1, 18, 324), n), walks=n > 6144)


@pytest.mark.parametrize("n", [1, 513, 4096, 4097])
def test_fp64(gpu, orc, n):
    solve(gpu, orc, *banded(n, [o for o in (1, 64) if o < n], n, dtype=np.float64), tol=1e-10,
          walks=n > 4096)


def test_guess(gpu, orc):
    JA, IA, V = banded(3000, (1, 55), 3)
    g = np.random.default_rng(1).standard_normal(3000).astype(np.float32)
    solve(gpu, orc, JA, IA, V, guess=g, walks=False)


def test_offset_at_and_beyond_the_guard(gpu, orc):
    solve(gpu, orc, *banded(4000, (1, 1024), 5), walks=False)
    solve(gpu, orc, *banded(4000, (1, 1025), 5), walks=True)


def test_walks_what_does_not_fit(gpu, orc):
    # more diagonals than the mean row length (rows drop most of them), beside
    # the register form and in a launch of its own
    for n in (1500, 3000):
        solve(gpu, orc, *banded(n, (1, 7, 50, 51, 52, 300), 6, drop=0.7), walks=True)
    JA, IA, V = banded(3000, (1, 50), 7)
    s = slice(JA[1234], JA[1235])
    IA[s], V[s] = IA[s][::-1].copy(), V[s][::-1].copy()
    solve(gpu, orc, JA, IA, V, walks=True)


def batch(cm):
    """Systems that fit the registers, one that does not, one empty."""
    parts = [banded(300, (1, 17), 1), banded(2500, (1, 50), 2), banded(40, (1,), 3),
             banded(700, (1, 3, 9, 30, 31, 200), 4, drop=0.7), banded(1, (), 5)]
    off, JAs, IAs, Vs, nnz = [0], [], [], [], 0
    for JA, IA, V in parts:
        JAs.append(JA[:-1] + nnz)
        IAs.append(IA + off[-1])
        Vs.append(V)
        off.append(off[-1] + JA.size - 1)
        nnz += IA.size
    off = np.array(off[:2] + [off[1]] + off[2:], np.int32)  # system 1 has no rows
    JA = np.concatenate(JAs + [[nnz]]).astype(np.int32)
    IA, V = np.concatenate(IAs).astype(np.int32), np.concatenate(Vs)
    return parts, off, JA, IA, V


def test_batch_of_both_forms(gpu, orc):
    cm = gpu
    from cumat_amd.solvers import pcg_batched
    parts, off, JA, IA, V = batch(cm)
    n = int(off[-1])
    b = np.random.default_rng(0).uniform(-1, 1, n).astype(np.float32)
    d = cm.DeviceArray.from_numpy
    cm.reset_counters()
    x, its, errs = cm.DeviceArray(n), cm.DeviceArray(off.size - 1, dtype=np.int32), cm.DeviceArray(off.size - 1)
    pcg_batched(d(off), d(JA), d(IA), d(V), d(b), x, 1e-5, 4000, its, errs)
    assert cm.counters()["CgWalk"] == 1
    x, its, errs = x.numpy(), its.numpy(), errs.numpy()
    for s, (JAs_, IAs_, Vs_) in zip([0, 2, 3, 4, 5], parts):
        r = slice(off[s], off[s + 1])
        _, it, _ = orc.pcg(JAs_, IAs_, Vs_, b[r], off[s + 1] - off[s], tol=1e-5, max_iter=4000)
        assert errs[s] <= 1e-5 and abs(its[s] - it) <= 2 + it // 20
        y = np.add.reduceat(Vs_.astype(np.float64) * x[r].astype(np.float64)[IAs_], JAs_[:-1])
        bound = 1e-5 + (1 + its[s]) * 2.0 ** -23 * 4 * np.abs(Vs_).max() * np.linalg.norm(x[r]) / np.linalg.norm(b[r])
        assert np.linalg.norm(b[r] - y) / np.linalg.norm(b[r]) <= bound


def test_left_systems_behind_a_graph(gpu):
    """The walking kernel follows every replay, and reports an invalid pattern."""
    cm = gpu
    from cumat_amd.solvers import pcg_batched
    parts, off, JA, IA, V = batch(cm)
    n, S = int(off[-1]), off.size - 1
    d = cm.DeviceArray.from_numpy
    fixed = [d(off), d(JA), d(IA), d(V)]
    b, x, its, errs = cm.DeviceArray(n), cm.DeviceArray(n), cm.DeviceArray(S, dtype=np.int32), cm.DeviceArray(S)
    for seed in range(3):
        new = d(np.random.default_rng(seed).uniform(-1, 1, n).astype(np.float32))
        b.copy_from(new)
        pcg_batched(*fixed, b, x, 1e-5, 4000, its, errs, use_graph=True)
        x2, its2, errs2 = cm.DeviceArray(n), cm.DeviceArray(S, dtype=np.int32), cm.DeviceArray(S)
        pcg_batched(*fixed, new, x2, 1e-5, 4000, its2, errs2)
        for got, ref in ((x, x2), (its, its2), (errs, errs2)):
            assert got.numpy().tobytes() == ref.numpy().tobytes()
    # system 4 walks; a column of its last row leaves it
    bad = IA.copy()
    bad[JA[off[5]] - 1] = off[5]
    with pytest.raises(cm.capi.CumatArgError):
        pcg_batched(fixed[0], fixed[1], d(bad), fixed[3], b, x, 1e-5, 4000, its, errs)
    it, er = its.numpy().ravel(), errs.numpy().ravel()
    assert it[4] == -1 and np.isnan(er[4])
    assert np.all(er[[0, 2, 3, 5]] <= 1e-5)
