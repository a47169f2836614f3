"""Generated kernels for memory that lies across the evaluation's order:
component-wise programs with transposed leaves (64 x 64 tiles, cwise_tile.hip)
and reductions along strided axes (lanes along the kept axes, rxcol.hip). Both
keep the interpreter's bits, signed zeros and NaN included."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def both(cm, fn, reset=True):
    """fn's result by the interpreter and by the generated kernels."""
    out = []
    for mode in (0, 2):
        old = cm.jit_mode(mode)
        try:
            if reset:
                cm.reset_counters()
            before = cm.counters()["JitLaunch"]
            out.append(fn())
            assert cm.counters()["JitLaunch"] - before == mode // 2
        finally:
            cm.jit_mode(old)
    assert out[0].tobytes() == out[1].tobytes()
    return out[1]


def data(shape, dtype, seed):
    rng = np.random.default_rng(seed)
    if dtype == np.int32:
        return rng.integers(-2000, 2000, shape).astype(dtype)
    a = rng.standard_normal(shape).astype(dtype)
    a.reshape(-1)[:: 97] = -0.0
    return a


@pytest.mark.parametrize("shape", [(1, 32, 32), (3, 33, 65), (1, 63, 64), (17, 64, 64), (16, 65, 129), (2, 127, 40),
                                   (1, 31, 200)])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
@pytest.mark.parametrize("row_major", [False, True])
def test_transposed_leaves(gpu, shape, dtype, row_major):
    cm = gpu
    B, R, C = shape
    a, t = data((B, R, C), dtype, 1), data((B, C, R), dtype, 2)
    o = data((B, R, C), dtype, 3)
    A = cm.DeviceArray.from_numpy(a, row_major=row_major)
    T = cm.DeviceArray.from_numpy(t, row_major=row_major)
    O = cm.DeviceArray.from_numpy(o, row_major=not row_major)  # the other layout: transposed as well
    tt = np.transpose(t, (0, 2, 1))
    for mode, expect in ((cm.capi.ASSIGN, a + tt - o), (cm.capi.ADD, a + (a + tt - o))):
        def run():
            D = cm.DeviceArray.from_numpy(a, row_major=row_major)
            cm.assign(D, A.expr() + T.expr().T - O.expr(), mode=mode)
            return D.numpy(logical=True)
        got = both(cm, run)
        assert np.array_equal(got, expect)


def test_transposed_comparison_into_bool(gpu):
    cm = gpu
    a = data((5, 70, 70), np.float32, 4)
    A = cm.DeviceArray.from_numpy(a)

    def run():
        D = cm.DeviceArray(70, 70, 5, dtype=np.bool_)
        cm.assign(D, A.expr() < A.expr().T)
        return D.numpy(logical=True)
    assert np.array_equal(both(cm, run), a < np.transpose(a, (0, 2, 1)))


def reduce_both(cm, a, b, axis, op, row_major=False):
    """sum / min / ... of a * b (b broadcast), both ways."""
    A = cm.DeviceArray.from_numpy(a, row_major=row_major)
    Bv = cm.DeviceArray.from_numpy(b)
    return both(cm, lambda: cm.reduce(A.expr() * Bv, op, axis).numpy(logical=True))


# kept rows across a wavefront, reduced columns across a thread's elements, a
# row of 16 threads, a wavefront, a pass and several passes
@pytest.mark.parametrize("kept", [16, 63, 64, 65, 4200])
@pytest.mark.parametrize("length", [1, 3, 4, 5, 8, 9, 127, 128, 129, 513, 2048, 2049, 9000])
def test_column_reduction(gpu, kept, length):
    cm = gpu
    if kept * length > 1 << 23:
        kept = 1100
    a, b = data((1, kept, length), np.float32, kept), data((1, 1, length), np.float32, length)
    got = reduce_both(cm, a, b, cm.capi.AXIS_COL, "sum")
    x = a.astype(np.float64) * b
    # pairwise over 256 threads, each a chain of length / 256 terms: far inside sqrt(length) eps
    bound = 2.0 ** -23 * np.sqrt(length + 8.0) * np.abs(x).sum(axis=2, keepdims=True)
    assert np.all(np.abs(got - x.sum(axis=2, keepdims=True)) <= bound)


@pytest.mark.parametrize("axis", [1, 2, 4, 5, 6])
@pytest.mark.parametrize("op", ["sum", "prod", "min", "max"])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_axes_and_operators(gpu, axis, op, dtype):
    cm = gpu
    a, b = data((9, 70, 130), dtype, axis), data((1, 70, 1), dtype, 7)
    if op == "prod":
        a, b = (1 + a * 1e-3).astype(dtype), (1 + b * 1e-3).astype(dtype)
    if dtype != np.int32 and op in ("min", "max"):
        a[2, 3, 5] = np.nan
        a[1] = -0.0
        a[5] = 0.0
    for row_major in (False, True):
        reduce_both(cm, a, b, axis, op, row_major)


@pytest.mark.parametrize("length", [1, 4, 5, 40, 128, 129])
@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_many_short_segments(gpu, length, dtype):
    """Contiguous segments of a flat program, on both sides of the rule."""
    cm = gpu
    a, b = data((1, length, 40000), dtype, 5), data((1, length, 40000), dtype, 6)
    A, Bv = cm.DeviceArray.from_numpy(a), cm.DeviceArray.from_numpy(b)
    got = both(cm, lambda: cm.reduce((A.expr() - Bv).cwiseAbs2(), "sum", cm.capi.AXIS_ROW).numpy(logical=True))
    x = (a.astype(np.float64) - b) ** 2
    assert np.all(np.abs(got - x.sum(axis=1, keepdims=True)) <= np.finfo(dtype).eps * (length + 4) * x.sum(axis=1, keepdims=True))


def test_bool_result(gpu):
    cm = gpu
    a = data((3, 100, 90), np.float32, 8)
    A = cm.DeviceArray.from_numpy(a)
    for op, ref in (("all", np.all), ("any", np.any)):
        got = both(cm, lambda: cm.reduce(A.expr() > cm.as_expr(np.float32(-2.5)), op, cm.capi.AXIS_COL).numpy(logical=True))
        assert np.array_equal(got, ref(a > -2.5, axis=2, keepdims=True))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
def test_short_segments_share_a_kernel(gpu, dtype):
    """A flat program's kernel serves every size: a program whose sizes change
    compiles once."""
    cm = gpu
    cm.reset_counters()
    for length, count in ((40, 40000), (41, 40001), (100, 33000), (9, 33333), (40, 40000)):
        a, b = data((3, length, count), dtype, 11), data((3, length, count), dtype, 12)
        A, Bv = cm.DeviceArray.from_numpy(a), cm.DeviceArray.from_numpy(b)
        ex = (A.expr() * 1.25 - Bv).cwiseAbs2()  # a program of this test alone
        got = both(cm, lambda: cm.reduce(ex, "sum", cm.capi.AXIS_ROW).numpy(logical=True), reset=False)
        x = (a.astype(np.float64) * 1.25 - b) ** 2
        assert np.all(np.abs(got - x.sum(axis=1, keepdims=True)) <= np.finfo(dtype).eps * (length + 6) * x.sum(axis=1, keepdims=True))
    assert cm.counters()["JitCompile"] == 1


@pytest.mark.parametrize("diagonal_first", [False, True])
def test_diagonal_leaf_after_its_broadcast_twin(gpu, diagonal_first):
    """v.asDiagonal() has the strides of v broadcast over the columns: neither
    may run the kernel generated for the other."""
    cm = gpu
    n, batches = 64, 512 + diagonal_first  # 32768 and more short folds; a shape of its own for each order
    a, v = data((batches, n, n), np.float32, 9), data((1, n, 1), np.float32, 10)
    A, V = cm.DeviceArray.from_numpy(a), cm.DeviceArray.from_numpy(v)
    exact = a.astype(np.float64) * v
    cases = [(V.expr(), exact), (V.expr().asDiagonal(), exact * np.eye(n))]
    for leaf, x in reversed(cases) if diagonal_first else cases:
        got = cm.reduce(A.expr() * leaf, "sum", cm.capi.AXIS_COL).numpy(logical=True)
        bound = 2.0 ** -23 * (n + 4) * np.abs(x).sum(axis=2, keepdims=True)
        assert np.all(np.abs(got - x.sum(axis=2, keepdims=True)) <= bound)
