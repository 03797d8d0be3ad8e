"""GPU parity of column reductions (a strided axis with unit-stride outputs) at the edges of their
kernels: whole-row steps over narrow rows (the period of odd row lengths, masked last rounds, column
strips, several tiles folded by a second launch), one lane per output vector, and rows of odd length
in the 64-lane column kernel.  Bounds as in test_gpu_reduce.py."""
import numpy as np
import pytest

import musapy_amd as ms
from musapy_amd import _core
from oracle import reference as R
from tests.conftest import assert_bits_equal
from tests.test_gpu_reduce import check_reduce, dev

pytestmark = pytest.mark.gpu
RNG = np.random.default_rng(4711)

# (shape, axis): what the shape reaches; the kernel depends on the type and the op too (ROUTES below pins some)
SHAPES = [
    ((7, 2), 0), ((2, 3), 0), ((1, 5), 0),                      # a slice of less than one step
    ((50000, 2), 0), ((20000, 3), 0), ((9001, 37), 0),          # short periods, several tiles
    ((1500, 511), 0), ((1501, 257), 0),                         # periods near a whole block
    ((4097, 96), 0), ((300, 700), 0), ((257, 640), 0),          # column strips, the last one narrower
    ((900, 1024), 0), ((900, 1020), 0), ((301, 1025), 0),       # either side of 4 KB rows (f32)
    ((130, 4099), 0), ((3, 100, 130), 1),                       # odd rows of the column kernel
    ((9, 500, 5), 1), ((40, 33, 7), 1), ((300, 6, 13), 1),      # many short slices
    ((70, 5, 2001), 1), ((2, 3, 70001), 1),                     # one lane per output vector
]


def values(kind, dt, shape):
    if dt == np.int64:
        return RNG.integers(-1000, 1000, shape).astype(np.int64)
    x = RNG.uniform(0.999, 1.001, shape) if kind == "prod" else RNG.standard_normal(shape)
    if dt in (np.complex64, np.complex128):
        x = x + 1j * RNG.standard_normal(shape) * (1e-3 if kind == "prod" else 1)
    return x.astype(dt)


KINDS = [(k, d) for d in (np.float32, np.float64, np.int64) for k in ("sum", "mean", "max", "argmin")]
KINDS += [("prod", np.float32), ("min", np.float32), ("argmax", np.float64)]
KINDS += [(k, d) for d in (np.complex64, np.complex128) for k in ("sum", "mean")]


@pytest.mark.parametrize("kind,dt", KINDS, ids=[f"{k}-{np.dtype(d).name}" for k, d in KINDS])
def test_column_shapes(kind, dt):
    for shape, axis in SHAPES:
        check_reduce(kind, values(kind, dt, shape), axis)


@pytest.mark.parametrize("kind", ["max", "min", "argmax", "argmin"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_column_ordered_semantics(kind, dt):
    """Ties, both zeros, a NaN in row 0 (absorbs the column), later NaNs, all-NaN columns, infinities."""
    for shape, axis in SHAPES:
        x = RNG.integers(-2, 3, shape).astype(dt)
        y = np.moveaxis(x, axis, 0)
        n = y.shape[0]
        y[n // 2][..., 1::3] = np.nan
        y[0][..., ::5] = np.nan
        y[-1][..., 2::7] = -0.0
        if n > 2:
            y[1:, ..., -1] = np.nan
            y[0][..., -1] = -np.inf
        check_reduce(kind, x, axis)
    z = np.full((9001, 37), np.nan, dt)
    z[0] = np.inf if kind.endswith("min") else -np.inf
    check_reduce(kind, z, 0)


@pytest.mark.parametrize("kind", ["sum", "max", "argmin"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_column_views(kind, dt):
    """Rows that are not contiguous, reversed rows of the axis, and bases off 16-byte alignment."""
    base = RNG.standard_normal((3001, 133)).astype(dt)
    B = dev(base)
    for lo, hi in ((0, 64), (1, 65), (3, 103), (5, 42), (2, 133)):
        check_reduce(kind, np.ascontiguousarray(base[:, lo:hi]), 0, gpu_x=ms.slice(B, [(0, 3001, 1), (lo, hi, 1)]))
        check_reduce(kind, np.ascontiguousarray(base[1::2, lo:hi]), 0, gpu_x=ms.slice(B, [(1, 3001, 2), (lo, hi, 1)]))
    check_reduce(kind, np.ascontiguousarray(base[::-1]), 0, gpu_x=ms.flip(B, 0))
    flat = RNG.standard_normal(3001 * 37 + 1).astype(dt)
    F = dev(flat)
    view = ms.slice(F, [(1, flat.size, 1)])  # 4 or 8 bytes past 16-byte alignment
    check_reduce(kind, flat[1:], None, gpu_x=view)


def test_column_results_repeat():
    """The same bits on every call, and with other reductions on the workspace in between."""
    x = RNG.standard_normal((40001, 37)).astype(np.float32)
    X = dev(x)
    first = [ms.sum(X, axis=0).numpy(), ms.argmax(X, axis=0).numpy()]
    for _ in range(3):
        ms.sum(X)
        assert_bits_equal(ms.sum(X, axis=0).numpy(), first[0], "sum")
        ms.max(X, axis=(0, 1))
        assert_bits_equal(ms.argmax(X, axis=0).numpy(), first[1], "argmax")
    assert_bits_equal(first[1], R.reduce(x, "argmax", 0), "argmax against the oracle")


# ---- unit-stride rows that start and end anywhere ----
@pytest.mark.parametrize("kind,dt", KINDS, ids=[f"{k}-{np.dtype(d).name}" for k, d in KINDS])
def test_row_lengths(kind, dt):
    """Every number of lanes per row with rows that end inside, at and after a vector (many short
    rows), and the last round of the wave, block and tiled kernels."""
    for shape in ((300001, 1), (140001, 3), (300003, 4), (140001, 5), (70001, 9), (70003, 16), (33001, 31),
                  (17001, 67), (9001, 130), (9001, 257), (4500, 513), (300, 1013), (70, 4097), (40, 8195),
                  (16, 16384), (3, 70001), (5, 40003)):
        if dt not in (np.float32, np.int64) and shape[0] > 20000:
            continue
        check_reduce(kind, values(kind, dt, shape), 1)


@pytest.mark.parametrize("kind", ["sum", "max", "argmin"])
@pytest.mark.parametrize("dt", [np.float32, np.float64])
def test_row_views_and_ordered_semantics(kind, dt):
    base = RNG.integers(-2, 3, (9001, 261)).astype(dt)
    if kind != "sum":
        base[::5, 0] = np.nan
        base[1::3, 100] = np.nan
        base[2::7, 1:] = np.nan
        base[3::7, -1] = -0.0
    B = dev(base)
    check_reduce(kind, base, 1)
    for lo, hi, step in ((1, 36, 1), (0, 133, 1), (3, 260, 1), (2, 258, 1), (0, 261, 3)):
        check_reduce(kind, np.ascontiguousarray(base[:, lo:hi:step]), 1,
                     gpu_x=ms.slice(B, [(0, 9001, 1), (lo, hi, step)]))
    long = RNG.integers(-2, 3, (5, 70003)).astype(dt)
    if kind != "sum":
        long[0, 0], long[1, -1] = np.nan, np.nan
    check_reduce(kind, np.ascontiguousarray(long[:, 1:]), 1, gpu_x=ms.slice(dev(long), [(0, 5, 1), (1, 70003, 1)]))


# (shape, axis, kind): kernel, whether its rows are split into tiles, column strips (f32)
ROUTES = [
    ((20011, 37), 0, "max", "spans", True, 1), ((20011, 37), 0, "mean", "spans", True, 1),
    ((40, 600, 37), 1, "argmin", "spans", False, 1), ((300, 700), 0, "max", "spans", False, 44),
    ((300, 700), 0, "sum", "spans", False, 44), ((12000, 1020), 0, "sum", "spans", True, 1),
    ((4000, 9, 37), 1, "sum", "lanes", False, 1), ((4000, 9, 37), 1, "argmax", "lanes", False, 1),
    ((70, 30, 2001), 1, "mean", "lanes", False, 1), ((4097, 96), 0, "max", "columns", False, 1),
    ((900, 2048), 0, "sum", "columns", False, 1), ((8000, 2048), 0, "argmin", "columns", False, 1),
]


@pytest.mark.parametrize("shape,axis,kind,kernel,tiled,strips", ROUTES, ids=str)
def test_column_kernels(shape, axis, kind, kernel, tiled, strips):
    itemsize, order = 4, 0 if kind in ("sum", "mean") else 2
    steps = [int(np.prod(shape[i + 1:])) for i in range(len(shape))]
    r = _core._route_columns(list(shape), steps, axis, itemsize, order)
    assert (r["kind"], r["tiles"] > 1, r["strips"]) == (kernel, tiled, strips)
    check_reduce(kind, values(kind, np.float32, shape), axis)


# ---- cumsum down the columns ----
SCAN_SHAPES = [
    ((63, 5), 0), ((64, 3), 0), ((384, 70), 0),                    # one lane per column, in order
    ((385, 64), 0), ((511, 65), 0), ((513, 3), 0),                 # one tile; two; fewer columns than a vector
    ((2049, 1), 0), ((3000, 2), 0), ((2600, 7), 0),                # thin arrays, claimed tiles
    ((1025, 513), 0), ((700, 1030), 0), ((2305, 130), 0),          # strips: a multiple of 8 or not, ragged
    ((3, 900, 33), 1), ((2, 3, 600, 18), 2), ((9, 400, 66), 1),    # outer dims
]


@pytest.mark.parametrize("dt", [np.float32, np.float64, np.int64])
def test_column_scan_shapes(dt):
    tol = {np.float32: 1e-5, np.float64: 1e-12}.get(dt)
    for shape, axis in SCAN_SHAPES:
        x = values("sum", dt, shape)
        got = ms.cumsum(dev(x), axis=axis).numpy()
        want = R.cumsum(x, axis)
        what = f"cumsum {np.dtype(dt).name} {shape} axis {axis}"
        if tol is None or shape[axis] <= 384:  # short axes keep the order of the reference
            assert_bits_equal(got, want, what)
        else:
            assert np.all(np.abs(got - want) <= tol * np.cumsum(np.abs(x.astype(np.float64)), axis=axis)), what
        for _ in range(2):
            assert_bits_equal(ms.cumsum(dev(x), axis=axis).numpy(), got, what + " again")


def test_column_scan_views_and_specials():
    base = RNG.integers(-100, 100, (1500, 90)).astype(np.int64)
    B = dev(base)
    assert_bits_equal(ms.cumsum(ms.flip(B, 0), axis=0).numpy(), np.cumsum(base[::-1], 0), "reversed axis")
    assert_bits_equal(ms.cumsum(ms.slice(B, [(1, 1500, 2), (3, 88, 1)]), axis=0).numpy(),
                      np.cumsum(base[1:1500:2, 3:88], 0), "every second row of some columns")
    for dt in (np.float32, np.float64):
        x = RNG.random((1300, 40)).astype(dt)
        x[700, 3] = np.inf
        x[900, 4] = np.nan
        x[10, 5], x[1200, 5] = np.inf, -np.inf
        x[:, 6] = -0.0
        got, want = ms.cumsum(dev(x), axis=0).numpy(), R.cumsum(x, 0)
        assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
        ok = np.isfinite(want)
        assert np.all(np.abs(got[ok] - want[ok]) <= 1e-5 * want[ok])
        assert not np.signbit(got[:, 6]).any()
