"""GPU parity of arrays large enough for streaming loads (32 MB of input) and stores (32 and 64 MB of output),
which smaller arrays never reach: operands that are broadcast, off a line or share their lines, and casts of
narrow elements.  Elementwise results and casts are exact."""
import numpy as np
import pytest

import musapy_amd as ms
from tests.conftest import assert_bits_equal
from tests.test_gpu_unaligned import dev, values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_binary_operands(dt):
    rows, cols = 4099, 4096 if dt == np.float32 else 2048  # 64 MB
    x = values(dt, (rows, cols + 4))
    row, col = values(dt, (cols + 5,)), values(dt, (rows + 1, 1))
    X, ROW, COL = dev(x), dev(row), dev(col)
    whole, shifted = X[:, :cols], X[:, 1:cols + 1]
    for y, Y in ((row[5:], ROW[5:]), (col[1:], COL[1:]), (row[3], ROW[3])):
        y, Y = (y[:cols], Y[:cols]) if y.shape == (cols,) else (y, Y)
        assert_bits_equal(ms.sub(whole, Y).numpy(), x[:, :cols] - y, "x - y")
        assert_bits_equal(ms.sub(Y, shifted).numpy(), y - x[:, 1:cols + 1], "y - x")
    assert_bits_equal(ms.sub(shifted, whole).numpy(), x[:, 1:cols + 1] - x[:, :cols], "neighbours")
    f = x.reshape(-1)
    F = dev(f)
    n = f.size - 7
    for lo in (1, 4, 7):
        assert_bits_equal(ms.add(F[lo:lo + n], F[:n]).numpy(), f[lo:lo + n] + f[:n], "runs off a line")
        assert_bits_equal(ms.abs(F[lo:lo + n]).numpy(), np.abs(f[lo:lo + n]), "a run off a line")
    assert_bits_equal(ms.abs(X[:, 2:cols - 1]).numpy(), np.abs(x[:, 2:cols - 1]), "rows of a slice")


@pytest.mark.parametrize("src,dst", [("int8", "float64"), ("uint8", "float32"), ("int16", "float64"),
                                     ("float32", "float64"), ("float64", "float32")])
def test_casts(src, dst):
    n = (64 << 20) // np.dtype(dst).itemsize
    x = np.random.default_rng(3).integers(-100 if src[0] != "u" else 0, 100, n + 4).astype(src)
    X = dev(x)
    short = {"float64": "f64", "float32": "f32"}[dst]
    for lo, hi in ((0, n), (0, n + 1), (3, n + 4)):
        assert_bits_equal(ms.astype(X[lo:hi], short).numpy(), x[lo:hi].astype(dst), f"{src} -> {dst} [{lo}:{hi}]")


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_transposed_operand_on_lines(dt):
    r, k = 4096, 2048 if dt == np.float64 else 4128  # every row of both operands starts on a line
    a, b = values(dt, (r, k)), values(dt, (k, r))
    assert_bits_equal(ms.sub(dev(a), ms.transpose(dev(b))).numpy(), np.ascontiguousarray(a - b.T), "a - b.T")


# (shape, axis): streamed and numbered tiles on lines, and with odd rows; claimed tiles, more than a window of them;
# one lane per column with 16 rows and, many narrow slices, 32 rows of loads in flight
@pytest.mark.parametrize("shape,axis", [((8192, 4096), 0), ((8193, 4099), 0), ((12000, 1601), 0), ((450, 131072), 0),
                                        ((10000, 500, 5), 1), ((30000, 100, 7), 1)], ids=str)
@pytest.mark.parametrize("dt", [np.int64, np.float32, np.float64])
def test_column_scans(dt, shape, axis):
    if dt != np.float32 and shape[-1] > 64:
        shape = shape[:-1] + (shape[-1] // 2,)
    x = values(dt, shape)
    got = ms.cumsum(dev(x), axis=axis).numpy()
    want = np.cumsum(x, axis, dtype=dt if dt == np.int64 else np.float64 if dt == np.float32 else np.longdouble)
    if dt == np.int64:
        assert_bits_equal(got, want, "cumsum")
        return
    # any order of n additions is within n * u * sum |x| of the exact sum
    bound = shape[axis] * np.finfo(dt).eps / 2 * np.cumsum(np.abs(x), axis, dtype=np.float64)
    assert np.all(np.abs(got - want) <= bound * 1.001)
