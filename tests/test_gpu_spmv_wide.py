"""The CSR product of rows with more than 8 entries on average (windows of 512
entries per 64 rows) and of several vectors with shared values, at the edges of
the windows, chunks and groups; int32 exactly, floats against FP64."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def matrix(lengths, cols, seed, dtype):
    rng = np.random.default_rng(seed)
    JA = np.zeros(len(lengths) + 1, np.int32)
    JA[1:] = np.cumsum(lengths)
    IA = rng.integers(0, cols, JA[-1]).astype(np.int32)
    V = rng.integers(-50, 50, IA.size).astype(dtype) if dtype == np.int32 else rng.standard_normal(IA.size).astype(dtype)
    return JA, IA, V


def check(cm, lengths, cols, dtype, batches=1, mode=0, shared_x=False, seed=0):
    JA, IA, V = matrix(lengths, cols, seed, dtype)
    n = len(lengths)
    rng = np.random.default_rng(seed + 1)
    draw = (lambda m: rng.integers(-50, 50, m).astype(dtype)) if dtype == np.int32 else (
        lambda m: rng.standard_normal(m).astype(dtype))
    x, y = draw((1 if shared_x else batches) * cols), draw(batches * n)
    A = cm.SparseMatrix.from_csr(n, cols, JA, IA, V)
    Y = cm.DeviceArray.from_numpy(y, rows=n, batches=batches)
    X = cm.DeviceArray.from_numpy(x, rows=cols, batches=1 if shared_x else batches)
    A.matvec(X, out=Y, mode=mode)
    got = Y.numpy().reshape(batches, n)
    wide = np.int64 if dtype == np.int32 else np.float64
    rows = np.repeat(np.arange(n), np.diff(JA))
    for b in range(batches):
        terms = V.astype(wide) * x.reshape(-1, cols)[0 if shared_x else b].astype(wide)[IA]
        total, size = np.zeros(n, wide), np.zeros(n, wide)
        np.add.at(total, rows, terms)
        np.add.at(size, rows, np.abs(terms))
        base = y.reshape(batches, n)[b].astype(wide) * (mode == 1)
        if dtype == np.int32:
            assert np.array_equal(got[b], (total + base).astype(np.int32))
        else:
            # every term meets at most its row's length additions and one product rounding
            bound = np.finfo(dtype).eps * ((np.asarray(lengths) + 2) * size + np.abs(base))
            assert np.all(np.abs(got[b] - (total + base)) <= bound)


@pytest.mark.parametrize("rows", [1, 63, 64, 65, 1000])
@pytest.mark.parametrize("length", [9, 27, 32, 64, 127, 128, 129, 700])
def test_row_lengths(gpu, rows, length):
    check(gpu, [length] * rows, 5000, np.int32)
    check(gpu, [length] * rows, 5000, np.float32, mode=gpu.capi.ADD)


@pytest.mark.parametrize("dtype", [np.int32, np.float32, np.float64])
def test_ragged_rows(gpu, dtype):
    rng = np.random.default_rng(3)
    lengths = rng.integers(0, 60, 4321)
    lengths[1000:1100] = 0
    lengths[2000] = 5000  # its chunk goes row by row
    check(gpu, lengths, 9000, dtype)


@pytest.mark.parametrize("batches", [2, 3, 4, 5, 8])
@pytest.mark.parametrize("mean", [4, 12])
def test_vectors_together(gpu, batches, mean):
    rows = 64 * 16384 // batches + 17  # past the rule: groups of vectors
    lengths = np.random.default_rng(batches).integers(0, 2 * mean + 1, rows)
    check(gpu, lengths, 1000, np.int32 if batches % 2 else np.float32, batches=batches)


@pytest.mark.parametrize("batches", [2, 3, 4])
@pytest.mark.parametrize("mean", [4, 12])
@pytest.mark.parametrize("dtype", [np.float64, np.float32, np.int32])
def test_long_rows_and_vectors_together(gpu, batches, mean, dtype):
    """Chunks that go row by row for all vectors of a group: both sides of a
    wavefront and of four, a few entries to thousands."""
    rows = 64 * 16384 // batches + 3
    lengths = np.full(rows, mean, np.int64)
    lengths[64 * np.arange(12) + np.arange(12)] = [129, 255, 256, 257, 320, 511, 512, 513, 575, 1000, 1024, 4097]
    lengths[64 * 20: 64 * 21] = 300  # every row of a chunk
    lengths[-2:] = [700, 0]
    check(gpu, lengths, 1000, dtype, batches=batches, mode=gpu.capi.ADD if batches == 3 else 0)


@pytest.mark.parametrize("rows", [64 * 1500 - 64, 64 * 1500])
def test_rule_for_groups_of_windows(gpu, rows):
    """Both sides of the limit from which the vectors of windows go together."""
    lengths = np.random.default_rng(8).integers(1, 40, rows)
    lengths[77] = 100
    check(gpu, lengths, 1000, np.int32, batches=3)
    check(gpu, lengths, 1000, np.float64, batches=3)


def test_shared_vector_and_bf16_values(gpu):
    cm = gpu
    check(cm, [20] * 3000, 3000, np.float32, batches=3, shared_x=False)
    JA, IA, V = matrix([20] * 3000, 3000, 5, np.float32)
    bits = (V.view(np.uint32) >> 16).astype(np.uint16)  # truncated to bf16
    A = cm.SparseMatrix(cm.SparsityPattern(3000, 3000, JA, IA), cm.DeviceArray.from_numpy(bits))
    x = np.random.default_rng(6).integers(-8, 8, 3000).astype(np.float32)
    got = A.matvec(cm.DeviceArray.from_numpy(x)).numpy()
    v = (bits.astype(np.uint32) << 16).view(np.float32).astype(np.float64)
    terms = v * x[IA]
    want, size = (np.add.reduceat(t, JA[:-1]) for t in (terms, np.abs(terms)))
    assert np.all(np.abs(got - want) <= 2.0 ** -23 * 22 * size)


@pytest.mark.parametrize("dtype,limit", [(np.int32, 30), (np.float64, 44)])
def test_crowded_windows(gpu, dtype, limit):
    """Both sides of the limit on a chunk's mean where the wavefronts fill the chip."""
    lengths = np.full(64 * 3072, limit, np.int64)
    lengths[:64 * 1000: 64] += 1
    check(gpu, lengths, 500, dtype)


@pytest.mark.parametrize("length", [9, 20, 27, 32, 39, 48, 64])
@pytest.mark.parametrize("signs", [False, True])
def test_windows_lose_no_precision(gpu, length, signs):
    """The rms error of 20000 rows is no larger than row by row: a product per
    lane and the wavefront's tree, emulated here. 3 % for the sampling."""
    cm = gpu
    rows, cols, f = 20000, 4000, np.float32
    rng = np.random.default_rng(length)
    draw = rng.standard_normal if signs else rng.random
    JA = (np.arange(rows + 1) * length).astype(np.int32)
    IA = rng.integers(0, cols, rows * length).astype(np.int32)
    V, x = draw(IA.size).astype(f), draw(cols).astype(f)
    A = cm.SparseMatrix.from_csr(rows, cols, JA, IA, V)
    got = A.matvec(cm.DeviceArray.from_numpy(x)).numpy().reshape(-1)
    lanes = np.zeros((rows, 64), f)
    lanes[:, :length] = (V * x[IA]).reshape(rows, length)
    while lanes.shape[1] > 1:
        lanes = lanes[:, 0::2] + lanes[:, 1::2]
    terms = (V.astype(np.float64) * x[IA]).reshape(rows, length)
    rms = lambda y: np.sqrt(np.mean(((y - terms.sum(1)) / np.abs(terms).sum(1)) ** 2))
    assert rms(got) <= 1.03 * rms(lanes[:, 0])


@pytest.mark.parametrize("batches", [1, 2, 3, 5])
@pytest.mark.parametrize("width", [3, 8, 9, 27])
@pytest.mark.parametrize("dtype", [np.float32, np.float64, np.int32])
def test_ell_vectors_together(gpu, batches, width, dtype):
    """ELLPACK with padding, past the rule for groups of vectors: integer data, exact in every type."""
    cm = gpu
    rows, cols = 64 * 16384 // batches + 5, 777
    rng = np.random.default_rng(width)
    idx = rng.integers(-1, cols, (rows, width)).astype(np.int32)
    val = rng.integers(-9, 10, (rows, width)).astype(dtype)
    x = rng.integers(-9, 10, (batches, cols)).astype(dtype)
    A = cm.ELLMatrix(rows, cols, idx, val)
    got = A.matvec(cm.DeviceArray.from_numpy(x.reshape(-1), rows=cols, batches=batches)).numpy().reshape(batches, rows)
    for b in range(batches):
        want = np.where(idx >= 0, val * x[b][np.maximum(idx, 0)], 0).sum(axis=1)
        assert np.array_equal(got[b], want.astype(dtype))
