"""GPU parity of binary ops with one transposed operand: edges and remainders of every tile shape, the
transposed operand on either side, the other one unit-stride, broadcast along either dim or sliced, batches,
and the forms just outside the rule.  Elementwise results are exact."""
import numpy as np
import pytest

import musapy_amd as ms
from tests.conftest import assert_bits_equal
from tests.test_gpu_unaligned import dev, values

pytestmark = pytest.mark.gpu

# output shapes: narrow in either dim, one element around a tile of each shape, and enough for the large tile
SHAPES = [(1, 40), (7, 8), (8, 8), (8, 33), (16, 4099), (4099, 16), (31, 65), (33, 63), (300, 31), (257, 33),
          (130, 127), (2049, 2050)]


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.complex64, np.complex128])
@pytest.mark.parametrize("shape", SHAPES, ids=str)
def test_transposed_operand(dt, shape):
    r, k = shape
    bt, a = values(dt, (k, r)), values(dt, (r, k))
    T = ms.transpose(dev(bt))
    for y in (a, values(dt, (r, 1)), values(dt, (k,))):
        Y = dev(y)
        assert_bits_equal(ms.sub(Y, T).numpy(), np.ascontiguousarray(y - bt.T), "y - x.T")
        assert_bits_equal(ms.sub(T, Y).numpy(), np.ascontiguousarray(bt.T - y), "x.T - y")
    assert_bits_equal(ms.add(T, ms.transpose(dev(bt + bt))).numpy(), np.ascontiguousarray((bt + (bt + bt)).T), "both")
    if dt in (np.float32, np.float64):
        assert_bits_equal(ms.lt(dev(a), T).numpy().astype(bool), a < bt.T, "lt")


@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_views_and_batches(dt):
    b, r, k = 3, 133, 70
    x, y = values(dt, (b, k + 1, r + 2)), values(dt, (b, r, k + 3))
    X, Y = dev(x), dev(y)
    xt, yt = np.swapaxes(x[:, 1:, 1:r + 1], 1, 2), y[:, :, 2:k + 2]
    got = ms.sub(Y[:, :, 2:k + 2], ms.permute(X[:, 1:, 1:r + 1], (0, 2, 1)))
    assert_bits_equal(got.numpy(), yt - xt, "batched slices")
    got = ms.sub(Y[1, :, 2:k + 2], ms.permute(X[:, 1:, 1:r + 1], (0, 2, 1)))
    assert_bits_equal(got.numpy(), yt[1] - xt, "broadcast batch")
    got = ms.sub(ms.permute(ms.flip(X, 1), (2, 0, 1)), dev(np.ascontiguousarray(np.transpose(x, (2, 0, 1)))))
    assert_bits_equal(got.numpy(), np.transpose(x[:, ::-1], (2, 0, 1)) - np.transpose(x, (2, 0, 1)), "rotated, flipped")
