"""GPU parity of the elementwise kernels on rows and arrays that start anywhere: element-aligned vectors,
the partial last item of a row, flipped rows, and edge tiles of transposed views."""
import numpy as np
import pytest

import musapy_amd as ms
from tests.conftest import assert_bits_equal
from tests.test_gpu_reduce import dev

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(815)
# row lengths around one item (4 f32, 2 f64), one 512-lane piece and one pair of pieces
LENGTHS = [1, 2, 3, 4, 5, 7, 37, 1023, 1025, 2047, 2049, 4095, 4097, 4101, 8191]


def values(dt, shape):
    if np.dtype(dt).kind in "iu":
        return RNG.integers(0, 100, shape).astype(dt)
    x = RNG.standard_normal(shape)
    if np.dtype(dt).kind == "c":
        x = x + 1j * RNG.standard_normal(shape)
    return x.astype(dt)


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("L", LENGTHS)
def test_binary_rows(dt, L):
    rows = 5
    a, row, col = values(dt, (rows, L)), values(dt, (L,)), values(dt, (rows, 1))
    for x, y in ((a, row), (row, a), (a, col), (col, row)):
        assert_bits_equal(ms.sub(dev(x), dev(y)).numpy(), x - y, f"{L}")
    # neighbours along the row, and flipped against straight
    w = values(dt, (rows, L + 1))
    W = dev(w)
    got = ms.sub(ms.slice(W, [(0, rows, 1), (1, L + 1, 1)]), ms.slice(W, [(0, rows, 1), (0, L, 1)]))
    assert_bits_equal(got.numpy(), w[:, 1:] - w[:, :-1], f"shifted {L}")
    got = ms.add(ms.flip(W, 1)[:, :L], W[:, 1:])
    assert_bits_equal(got.numpy(), w[:, ::-1][:, :L] + w[:, 1:], f"flipped {L}")
    if dt in (np.float32, np.float64):
        assert_bits_equal(ms.lt(W[:, 1:], W[:, :-1]).numpy().astype(bool), w[:, 1:] < w[:, :-1], f"lt {L}")


@pytest.mark.parametrize("dt", [np.uint8, np.int32, np.float32, np.float64])
@pytest.mark.parametrize("n", [1, 15, 63, 64, 257, 1025, 4099])
def test_flat_and_unary(dt, n):
    v = values(dt, (n + 3,))
    V = dev(v)
    for s in (1, 2, 3):
        assert_bits_equal(ms.contiguous(V[s:]).numpy(), v[s:], f"copy from {s}")
        to = np.float32 if dt == np.float64 else np.float64
        assert_bits_equal(ms.astype(V[s:s + n], np.dtype(to).name).numpy(), v[s:s + n].astype(to), f"cast from {s}")
    m = values(dt, (5, n + 3))
    M = dev(m)
    assert_bits_equal(ms.contiguous(M[:, 1:]).numpy(), m[:, 1:], "rows")
    assert_bits_equal(ms.contiguous(ms.flip(M, 1)).numpy(), m[:, ::-1], "flip")
    if dt in (np.float32, np.float64):
        assert_bits_equal(ms.add(V[1:], V[:-1]).numpy(), v[1:] + v[:-1], "flat")
    if dt == np.float64:
        i = RNG.integers(-9, 9, n + 3)
        assert_bits_equal(ms.add(dev(i)[1:], V[:-1]).numpy(), i[1:] + v[:-1], "mixed")


@pytest.mark.parametrize("dt", [np.uint8, np.float32, np.float64, np.complex128])
@pytest.mark.parametrize("shape", [(127, 129), (129, 131), (257, 65), (33, 301), (301, 7), (5, 130), (3, 131, 133)])
def test_transposed_views(dt, shape):
    m = values(dt, shape)
    M, t = dev(m), (lambda x: np.swapaxes(x, -1, -2))
    axes = tuple(range(len(shape) - 2)) + (len(shape) - 1, len(shape) - 2)
    assert_bits_equal(ms.contiguous(ms.permute(M, axes)).numpy(), np.ascontiguousarray(t(m)), "whole")
    if len(shape) == 2:
        got = ms.contiguous(ms.transpose(ms.slice(M, [(1, shape[0], 1), (1, shape[1], 1)])))
        assert_bits_equal(got.numpy(), np.ascontiguousarray(m[1:, 1:].T), "slice")
