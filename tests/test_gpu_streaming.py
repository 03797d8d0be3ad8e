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
