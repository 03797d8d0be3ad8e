"""Rounding error of floating-point sums against extended precision, for the kernels that hold partial sums
in the element's own type.  The bound is twice the rounding model of n / 8 additions in each of 8 chains and
a tree over them: an addition errs by at most u = 2^-24 (2^-53) of its result, evenly spread (u / sqrt(3)
rms); for values around 1 the result is the number of terms so far, so the errors of a column of n add up to
u / sqrt(3) * sqrt(8 * (n / 8)^3 / 3 + (1/4 + 1/2 + 1) * n^2) at most, over a sum of n.  One chain of
400 additions measured 2.9e-7 in float32, above the bound of 1.4e-7."""
import numpy as np
import pytest

import musapy_amd as ms
from musapy_amd import _core
from tests.conftest import assert_bits_equal
from tests.test_gpu_reduce import dev

pytestmark = pytest.mark.gpu


def bound(dt, n):
    u = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    return 2 * u / np.sqrt(3) * np.sqrt(8 * (n / 8) ** 3 / 3 + 1.75 * n ** 2) / n


# (shape, axis): one lane per vector of outputs over a long axis, narrow and wide; one block per slice
SHAPES = [((33000, 400, 4), 1), ((520, 400, 260), 1), ((260, 400, 500), 1)]


@pytest.mark.parametrize("dt", [np.float32, np.float64])
@pytest.mark.parametrize("shape,axis", SHAPES, ids=str)
def test_column_sums(dt, shape, axis):
    if dt == np.float64:
        shape = shape[:-1] + (shape[-1] // 2,)
    rng = np.random.default_rng(99)
    x = rng.random(shape, dtype=dt)
    x += dt(0.5)
    want = np.sum(x, axis=axis, dtype=np.longdouble)
    X = dev(x)
    for got, w in ((ms.sum(X, axis=axis), want), (ms.mean(X, axis=axis), want / shape[axis])):
        err = np.linalg.norm((got.numpy() - w).astype(np.float64)) / np.linalg.norm(w.astype(np.float64))
        assert err <= bound(dt, shape[axis]), err


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_column_kernel_sums(dt):
    """The column kernel: 8 waves of chains over n / 32 sums of 4 rows, and a tree over the waves.  By the same
    model u / sqrt(3) * sqrt(8 * 16 * (n / 32)^3 / 3 + 6 * n + 1.75 * n^2) over n, 5.2e-8 in float32 for 400 rows;
    rows and waves one after the other come to 7.9e-8.  An addition errs by u of the power of two below its result, so
    the model is itself a bound: about 0.7 of it is expected, 3.8e-8 against 5.7e-8."""
    n, shape = 400, (80, 400, 1024 if dt == np.float32 else 512)
    itemsize = np.dtype(dt).itemsize
    assert _core._route_columns(list(shape), [n * shape[2], shape[2], 1], 1, itemsize, 0)["kind"] == "columns"
    x = np.random.default_rng(7).random(shape, dtype=dt)
    x += dt(0.5)
    want = np.sum(x, axis=1, dtype=np.longdouble)
    got = ms.sum(dev(x), axis=1).numpy()
    u = 2.0 ** -24 if dt == np.float32 else 2.0 ** -53
    model = u / np.sqrt(3) * np.sqrt(8 * 16 * (n / 32) ** 3 / 3 + 6 * n + 1.75 * n ** 2) / n
    err = np.linalg.norm((got - want).astype(np.float64)) / np.linalg.norm(want.astype(np.float64))
    assert err <= model, err


def tree(t):
    """Sums along the last axis, halves first: t[i] + t[i + n / 2] while n > 1."""
    while t.shape[-1] > 1:
        h = t.shape[-1] // 2
        t = t[..., :h] + t[..., h:]
    return t[..., 0]


@pytest.mark.parametrize("cols", [8, 9, 13, 33, 67])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_short_row_sums(dt, cols):
    """Many short rows: the same bits as a tree over each 16-byte vector and then over the lanes of the row
    (the vector that the end of a row cuts starts earlier, with zeros for the elements of the one before)."""
    V = 16 // np.dtype(dt).itemsize
    vecs = -(-cols // V)
    lanes = 1 << (vecs - 1).bit_length()
    rows = 524288 // lanes + 3
    x = np.random.default_rng(cols).random((rows, cols), dtype=dt) + dt(0.5)
    t = np.zeros((rows, lanes, V), dt)
    for v in range(vecs):
        n = min(V, cols - v * V)
        t[:, v, V - n:] = x[:, v * V:v * V + n]
    want = tree(tree(t))
    assert_bits_equal(ms.sum(dev(x), axis=1).numpy(), want, f"{np.dtype(dt).name} rows of {cols}")
