"""Reductions of stored arrays whose kept axis is the contiguous one, at the
shapes where the kernels change: few kept elements (several rows per wavefront),
short folds (a thread per output), long folds with many partials; all types."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DTYPES = [np.float32, np.float64, np.int32, np.bool_]


def check(cm, shape, axis, dtype, op="sum"):
    B, R, C = shape
    rng = np.random.default_rng(R + C + B)
    if dtype == np.bool_:
        a, op = rng.uniform(size=shape) < 0.999, "all"
    elif dtype == np.int32:
        a = rng.integers(-1000, 1000, shape).astype(dtype)
    else:
        a = rng.uniform(0, 1, shape).astype(dtype)
    got = cm.reduce(cm.DeviceArray.from_numpy(a), op, axis).numpy(logical=True)
    dims = tuple(d for d, bit in ((1, 1), (2, 2), (0, 4)) if axis & bit)
    if dtype == np.bool_:
        assert np.array_equal(got, a.all(axis=dims, keepdims=True))
    elif dtype == np.int32:
        f = {"sum": np.sum, "min": np.min, "max": np.max}[op]
        assert np.array_equal(got, f(a.astype(np.int64), axis=dims, keepdims=True).astype(np.int32))
    else:
        want = a.astype(np.float64).sum(axis=dims, keepdims=True)
        n = a.size / want.size
        # positive terms: a chain of at most 2048 of them, then trees
        assert np.all(np.abs(got - want) <= np.finfo(dtype).eps * (min(n, 2048) + 30) * want)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [2, 3, 8, 31, 32, 33])
@pytest.mark.parametrize("cols", [63, 64, 65, 1000, 70001])
def test_few_kept_elements(gpu, dtype, rows, cols):
    check(gpu, (1, rows, cols), 2, dtype)
    check(gpu, (5, rows, cols // 5), 2, dtype)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("batches", [2, 3, 7, 8, 9, 61])
def test_short_folds(gpu, dtype, batches):
    check(gpu, (batches, 517, 519), 4, dtype)  # one output more than a thread each for 256 CUs x 1024


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(40, 100, 700), (40, 1024, 257), (7, 64, 5003), (3, 260, 9001)])
def test_long_folds(gpu, dtype, shape):
    check(gpu, shape, 6, dtype)
    check(gpu, shape, 2, dtype)


@pytest.mark.parametrize("op", ["min", "max"])
def test_extrema(gpu, op):
    for shape, axis in (((1, 5, 9000), 2), ((3, 600, 601), 4), ((9, 100, 900), 6)):
        check(gpu, shape, axis, np.int32, op)


def strided(x, k, step):
    """A lane's fold of x[k], x[k + step], ...: groups of four, then one by one."""
    acc = np.zeros_like(x[0])
    while k + 3 * step < len(x):
        acc = acc + ((x[k] + x[k + step]) + (x[k + 2 * step] + x[k + 3 * step]))
        k += 4 * step
    while k < len(x):
        acc = acc + x[k]
        k += step
    return acc


def chain(parts):
    r = parts[0]
    for v in parts[1:]:
        r = r + v
    return r


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("batches", [2, 3, 5, 8, 12, 13, 14, 15, 16, 17, 29, 32, 61, 100])
def test_short_folds_keep_four_partials(gpu, dtype, batches):
    # the order of four wavefronts splitting the fold, one output per thread
    a = np.random.default_rng(batches).normal(size=(batches, 517, 519)).astype(dtype)
    got = gpu.reduce(gpu.DeviceArray.from_numpy(a), "sum", 4).numpy(logical=True)
    assert np.array_equal(got[0], chain([strided(a, w, 4) for w in range(4)]))


@pytest.mark.parametrize("dtype", [np.float32, np.float64])
@pytest.mark.parametrize("rows", [2, 3, 5, 8, 31, 32])
@pytest.mark.parametrize("cols", [64, 100, 255])
def test_few_kept_elements_fold_by_halves(gpu, dtype, rows, cols):
    # more batches than blocks wanted, so that a fold is one block's
    a = np.random.default_rng(cols + rows).normal(size=(2100, rows, cols)).astype(dtype)
    got = gpu.reduce(gpu.DeviceArray.from_numpy(a), "sum", 2).numpy(logical=True)[:, :, 0]
    x, per = np.moveaxis(a, 2, 0), 64 // rows
    r = [chain([strided(x, w * per + s, 4 * per) for w in range(4)]) for s in range(per)]
    while len(r) > 1:
        h = (len(r) + 1) // 2
        r = [r[i] + r[i + h] if i + h < len(r) else r[i] for i in range(h)]
    assert np.array_equal(got, r[0])


def test_few_kept_elements_of_few_batches_lose_no_precision(gpu):
    """The rms error over 38400 folds of 180 rows is no larger than that of the
    general kernel's order (three blocks of four wavefronts), emulated here."""
    P, Q, K, f = 300, 32, 180, np.float32
    errors = [[], []]
    for seed in range(4):
        rng = np.random.default_rng(seed)
        # a random scale for every fold, so that no sum sits at a power of two
        a = (rng.uniform(0, 1, (P, Q, K)) * 2 ** rng.uniform(0, 1, (P, Q, 1))).astype(f)
        want = a.astype(np.float64).sum(axis=2)
        x = np.moveaxis(a, 2, 0)
        general = chain([chain([strided(x[60 * s: 60 * s + 60], w, 4) for w in range(4)]) for s in range(3)])
        got = gpu.reduce(gpu.DeviceArray.from_numpy(a), "sum", 2).numpy(logical=True)[:, :, 0]
        for e, y in zip(errors, (got, general)):
            e.append((y - want) / want)
    rms = [np.sqrt(np.mean(np.square(e))) for e in errors]
    assert rms[0] <= rms[1]
