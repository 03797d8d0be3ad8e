"""GPU parity of reductions over integer arrays, which widen the elements inside the reduction instead
of casting the array first.  Integer results and indices are bit-exact; means of at most 32-bit
integers are the exact sum rounded once and divided, so they are within one rounding of any float64
sum below 2^53 (the inputs here stay below it), and int64/uint64 means keep the float64 bound."""
import numpy as np
import pytest

import musapy_amd as ms
from oracle import reference as R
from tests.conftest import assert_bits_equal
from tests.test_gpu_reduce import dev

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(8080)
TYPES = [np.int8, np.uint8, np.int16, np.uint16, np.int32, np.uint32, np.int64, np.uint64]
KINDS = ["sum", "prod", "max", "min", "mean", "argmax", "argmin"]

# (shape, axis): rows of every group size and their odd ends, strided rows, narrow and wide columns
# (flat spans, strips with a cut last vector, several tiles), one lane per vector, whole arrays
SHAPES = [
    ((300, 3), 1), ((300, 9), 1), ((70, 67), 1), ((33, 4099), 1), ((5, 70001), 1), ((2, 300007), 1),
    ((1000, 1), 0), ((5000, 3), 0), ((9000, 37), 0), ((700, 511), 0), ((2000, 513), 0), ((400, 2053), 0),
    ((3, 200, 129), 1), ((9, 40, 7), 1), ((60, 4, 5000), 1), ((1 << 20,), None), ((333333,), None), ((7,), None),
]


def values(dt, shape, kind):
    if kind == "prod":
        return RNG.integers(0 if np.dtype(dt).kind == "u" else -3, 4, shape).astype(dt)
    i = np.iinfo(dt)
    if np.dtype(dt).itemsize == 8:  # float64 sums of these are exact
        return RNG.integers(max(i.min, -(1 << 30)), 1 << 30, shape, dtype=np.int64).astype(dt)
    return RNG.integers(i.min, int(i.max) + 1, shape, dtype=np.int64).astype(dt)


def check(kind, x, axis, gpu_x=None):
    got = getattr(ms, kind)(dev(x) if gpu_x is None else gpu_x, axis=axis).numpy()
    want = R.reduce(np.ascontiguousarray(x), kind, axis)
    what = f"{kind} {x.dtype} {x.shape} axis={axis}"
    if kind == "mean":
        assert got.dtype == np.float64 and got.shape == want.shape, what
        assert np.all(np.abs(got - want) <= 1e-12 * np.mean(np.abs(x.astype(np.float64)), axis=axis)), what
    else:
        assert_bits_equal(got, want, what)


@pytest.mark.parametrize("kind", KINDS)
@pytest.mark.parametrize("dt", TYPES)
def test_int_reduce_shapes(kind, dt):
    for shape, axis in SHAPES:
        check(kind, values(dt, shape, kind), axis)


@pytest.mark.parametrize("dt", TYPES)
def test_int_reduce_ties_extremes_views(dt):
    i = np.iinfo(dt)
    for fill in (i.min, i.max):  # every element the lowest or highest value of the type
        x = np.full((700, 129), fill, dt)
        for kind in ("max", "min", "argmax", "argmin"):
            for axis in (0, 1, None):
                check(kind, x, axis)
    base = RNG.integers(0, 5, (600, 261)).astype(dt)
    B = dev(base)
    for kind in ("sum", "max", "argmin", "mean"):
        for axis in (0, 1, None):
            check(kind, base.T, axis, ms.transpose(B))
            check(kind, base[:, ::-1], axis, ms.flip(B, 1))
            check(kind, base[1::2, 3:200], axis, ms.slice(B, [(1, 600, 2), (3, 200, 1)]))
            check(kind, base[:, 1::3], axis, ms.slice(B, [(0, 600, 1), (1, 261, 3)]))
    check("sum", base.astype(dt).reshape(60, 10, 261), (0, 2))
    out = dev(np.zeros(600, np.int64))
    ms.sum(B, axis=1, out=out)
    assert_bits_equal(out.numpy(), R.reduce(base, "sum", 1), "out=")
