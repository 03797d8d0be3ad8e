"""Host-side logic of the product, on CPU: promotion, broadcasting, axis resolution, views,
launch planning and the 32-bit magic division used by the kernels.  Known answers come from
musapy's own unit tests (tests/golden/host_kats.json, regenerated by make_host_kats.py)."""
import json
import os

import numpy as np
import pytest

import musapy_amd as ms
from musapy_amd import _core
from oracle import reference as R

KATS = json.load(open(os.path.join(os.path.dirname(__file__), "golden", "host_kats.json")))
DTYPES = ["bool", "i8", "i16", "i32", "i64", "u8", "u16", "u32", "u64", "f16", "f32", "f64", "bf16", "c64", "c128"]


@pytest.mark.parametrize("case", KATS["promotion"], ids=lambda c: f"{c[0]}+{c[1]}:{c[2]}")
def test_promotion_kats(case):
    a, b, gpu, want = case
    assert _core._promote(a, b, gpu) == want
    assert R.promote(a, b, gpu) == want


def test_promotion_full_table_product_vs_oracle():
    for a in DTYPES:
        for b in DTYPES:
            for gpu in (False, True):
                assert _core._promote(a, b, gpu) == R.promote(a, b, gpu), (a, b, gpu)
                assert _core._promote(a, b, gpu) == _core._promote(b, a, gpu), (a, b, gpu)


def test_broadcast_kats():
    for shapes, want in KATS["broadcast_shape"]:
        if len(shapes) == 0:
            continue
        assert list(_core._broadcast_shape(shapes)) == want
    for shapes in KATS["broadcast_shape_error"]:
        with pytest.raises(ms.ShapeError):
            _core._broadcast_shape(shapes)
    for shape, target, want in KATS["broadcast_strides"]:
        strides = [int(s) for s in np.zeros(shape).strides] if shape else []
        strides = [s // 8 for s in strides]
        assert list(_core._broadcast_strides(shape, strides, target)) == want


def test_resolve_axes():
    assert _core._resolve_axes([-1, 0], 3) == [0, 2]
    with pytest.raises(ms.ShapeError):
        _core._resolve_axes([0, 0], 3)
    with pytest.raises(ms.ShapeError):
        _core._resolve_axes([5], 3)
    with pytest.raises(ms.ShapeError):
        _core._resolve_axes([-4], 3)


def test_layout_views():
    # layout.rs doc examples: flip / transpose / slice
    assert _core._layout_view([3, 4], "flip", 0) == ([3, 4], [-4, 1], 8)
    # an empty axis has no last element: the offset stays put instead of wrapping below zero
    assert _core._layout_view([0, 4], "flip", 0) == ([0, 4], [-4, 1], 0)
    assert _core._layout_view([2, 3], "transpose", None) == ([3, 2], [1, 3], 0)
    assert _core._layout_view([2, 3, 4], "transpose", [1, 2, 0]) == ([3, 4, 2], [4, 1, 12], 0)
    assert _core._layout_view([10, 6], "slice", ([2, 1], [9, 6], [3, 2])) == ([3, 3], [18, 2], 13)
    with pytest.raises(ms.ShapeError):
        _core._layout_view([2, 3], "transpose", [0, 0])
    with pytest.raises(ms.ShapeError):
        _core._layout_view([4], "slice", ([0], [5], [1]))


def test_cast_validation_matches_reference_rules():
    ok = ["i8", "i16", "i32", "i64", "u8", "u16", "u32", "u64", "f32", "f64"]
    for s in DTYPES:
        for d in DTYPES:
            try:
                R.validate_cast(s, d)
                want = True
            except R.OracleError:
                want = False
            try:
                _core._validate_cast(s, d)
                got = True
            except ms.DtypeError:
                got = False
            assert got == want, (s, d)
    assert set(ok) >= {"f32"}


def _walk(shape, strides):
    idx = np.indices(shape).reshape(len(shape), -1).T if shape else np.zeros((1, 0), int)
    return idx @ np.array(strides, dtype=np.int64) if shape else np.zeros(1, np.int64)


@pytest.mark.parametrize("shape,strides", [
    ([4096, 8192], [[1, 0], [0, 1]]),
    ([2, 3, 4], [[12, 4, 1], [12, 4, 1]]),
    ([2, 1, 3, 4], [[12, 12, 4, 1], [0, 0, 0, 1]]),
    ([5, 6, 7], [[1, 5, 30], [42, 7, 1]]),
    ([3, 4], [[-4, 1], [4, -1]]),
    ([1, 1], [[0, 0], [1, 1]]),
    ([], [[], []]),
])
def test_elementwise_plan_preserves_addresses(shape, strides):
    plan = _core._plan_elementwise(shape, strides)
    n = int(np.prod(shape)) if shape else 1
    assert plan["numel"] == n
    # the coalesced description visits exactly the same (output, input...) offsets in order
    out_c = [int(s) // 8 for s in np.zeros(shape).strides] if shape else []
    want = [_walk(shape, out_c)] + [_walk(shape, s) for s in strides]
    got = [_walk(plan["shape"], s) for s in plan["strides"]]
    for g, w in zip(got, want):
        assert np.array_equal(g, w)


def test_reduce_plan_kinds():
    assert _core._plan_reduce([8192, 8192], [8192, 1], 1)["kind"] == "row"
    p0 = _core._plan_reduce([8192, 8192], [8192, 1], 0)
    assert p0["kind"] == "col" and p0["tiles"] > 1
    p = _core._plan_reduce([16, 1024, 1024], [1048576, 1024, 1], 1)
    assert p["kind"] == "col" and p["oshape"] == [16, 1024]
    t = _core._plan_reduce([67108864], [1], 0)
    assert t["kind"] == "row" and t["tiles"] >= 256


def test_scan_plan_kinds():
    assert _core._plan_scan([1024, 65536], [65536, 1], 1)["kind"] == "row"
    assert _core._plan_scan([1024, 65536], [65536, 1], 0)["kind"] == "col"
    assert _core._plan_scan([8, 9], [1, 8], 1)["kind"] == "generic"


def test_grid_limits():
    """A grid dim holds fewer than 2^32 lanes, whatever the block size, and fewer than 2^31 blocks."""
    for lanes in (64, 128, 256, 512, 1024):
        most = min(2 ** 31 - 1, (2 ** 32 - 1) // lanes)
        assert _core._grid_fits(1, lanes) and _core._grid_fits(most, lanes)
        assert not _core._grid_fits(most + 1, lanes)
    assert not _core._grid_fits(8400000, 512)  # 16 x 16 transposed batches, one tile of 512 lanes each
    assert not _core._grid_fits(32768 * 128, 1024)  # cumsum of (32768, 262144, 2) along axis 1 in 2048-row tiles


def test_fastdiv_exact():
    rng = np.random.default_rng(5)
    divisors = [1, 2, 3, 5, 7, 10, 31, 64, 641, 1000, 4096, 6700417, 2**31 - 1, 2**31, 2**31 + 1, 2**32 - 1]
    divisors += rng.integers(1, 2**32, 40).tolist()
    for d in divisors:
        ns = [0, 1, d - 1, d, d + 1, 2**32 - 1, 2**31, 2**31 - 1] + rng.integers(0, 2**32, 500).tolist()
        ns = [n % 2**32 for n in ns]
        assert _core._fastdiv_check(d, ns) == [n // d for n in ns], d


def test_import_fails_loudly_without_device():
    # on a host without a GPU the package imports (the C ABI loads) but device work raises
    if _core.device_count() > 0:
        pytest.skip("a device is present")
    with pytest.raises(Exception):
        ms.array([1.0, 2.0])


# (shape, axis, element bytes, kind) -> kernel; kind 0 sums, 1 complex sums, 2 max / min / arg
COLUMN_ROUTES = [
    ([20000, 16, 8], 1, 4, 0, "lanes"), ([1000, 16, 512], 1, 4, 2, "lanes"), ([4000, 100, 300], 1, 4, 0, "lanes"),
    ([1000, 120003], 0, 4, 0, "columns"), ([1000, 300000], 0, 4, 0, "lanes"),
    ([256, 500, 512], 1, 4, 2, "columns"), ([4000, 100, 100], 1, 4, 0, "columns"),
    ([18, 5000, 600], 1, 4, 0, "spans"), ([8, 5000, 1000], 1, 4, 0, "columns"), ([10, 2100, 700], 1, 4, 2, "spans"),
    ([52, 263, 54], 1, 8, 2, "spans"), ([14, 500, 432], 1, 4, 0, "columns"), ([12, 2100, 371], 1, 8, 1, "spans"),
    ([300, 131072], 0, 4, 2, "columns"), ([1000003, 37], 0, 4, 0, "spans"), ([1000003, 37], 0, 8, 2, "spans"),
    ([131072, 384], 0, 4, 0, "spans"), ([64, 100, 1000], 1, 4, 0, "columns"), ([120, 2000, 1024], 1, 4, 0, "columns"),
    ([4000, 128], 0, 4, 2, "columns"), ([4000, 128], 0, 4, 0, "spans"), ([8, 600, 128], 1, 8, 1, "spans"),
    ([8, 600, 128], 1, 8, 0, "columns"), ([8, 4096, 1000], 1, 4, 0, "columns"), ([8192, 8192], 0, 4, 0, "columns"),
]


@pytest.mark.parametrize("shape,axis,es,kind,want", COLUMN_ROUTES, ids=str)
def test_column_reduction_routes(shape, axis, es, kind, want):
    strides = [int(np.prod(shape[i + 1:], dtype=np.int64)) for i in range(len(shape))]
    assert _core._route_columns(shape, strides, axis, es, kind)["kind"] == want


def test_column_strips_and_tiles():
    """Small inputs split by strips while one is at most one and a half rounds long, else by tiles."""
    assert _core._route_columns([600, 400], [400, 1], 0, 4, 0)["strips"] > 1
    r = _core._route_columns([3000, 100], [100, 1], 0, 4, 0)
    assert r["strips"] == 1 and r["tiles"] > 1


def test_short_row_routes():
    pays = _core._short_rows_pay  # (row length, vectors, accumulator bytes, ordered)
    assert all(pays(r, -(-r // 4), 4, False) for r in range(4, 513))
    assert not pays(33, 17, 16, True) and not pays(48, 24, 16, True) and pays(50, 25, 16, True)
    assert not pays(50, 25, 16, False) and pays(64, 32, 16, False) and not pays(5, 3, 16, True) and pays(6, 3, 16, True)


def test_ordered_rows_by_waves():
    waves = _core._ordered_waves  # (bytes of a row, rows)
    assert waves(16384, 16384) and waves(16384, 1000) and waves(28000, 1536) and waves(32000, 2048)
    assert not waves(24000, 500) and not waves(32000, 64) and not waves(32000, 16384)
    assert not waves(32768, 16384) and not waves(16380, 16384)


# which operands of a large f32 binary op stream (first, second, transposed tiles); the operands start at the given
# addresses, far apart unless `meet`
@pytest.mark.parametrize("shape,sa,sb,a,b,want", [
    ((1 << 24,), (1,), (1,), 0, 0, (1, 1, 1)), ((1 << 24,), (1,), (1,), 16, 0, (1, 1, 0)),  # runs
    ((1 << 24,), (1,), (0,), 4, 0, (1, 0, 0)), ((1 << 24,), (0,), (1,), 0, 0, (0, 1, 1)),  # a scalar
    ((20000, 4096), (4096, 1), (1, 0), 0, 0, (1, 0, 1)), ((20000, 4003), (4003, 1), (1, 0), 4, 0, (1, 0, 0)),  # a column
    ((20000, 4096), (4096, 1), (0, 1), 0, 4, (1, 0, 1)), ((20000, 4003), (4003, 1), (0, 1), 0, 0, (0, 0, 0)),  # a row
    ((20000, 4003), (0, 1), (4003, 1), 0, 0, (0, 0, 0)),
    ((20000, 4096), (4100, 1), (4100, 1), 0, 0, (1, 1, 0)),  # two slices
    ((20000, 4003), (4004, 1), (4004, 1), 0, "meet", (0, 0, 0)),  # neighbours in one array
    ((8192, 4096), (4096, 1), (1, 8192), 0, 0, (1, 1, 1)),  # transposed
], ids=str)
def test_binary_loads(shape, sa, sb, a, b, want):
    base = 1 << 32
    second = base + 4 if b == "meet" else base * 2 + b
    assert _core._binary_loads(shape, [sa, sb], 4, base + a, second) == [bool(w) for w in want]


# (P, L, elements of the output, element bytes) -> tile of a binary op with a transposed operand
@pytest.mark.parametrize("args,want", [
    ((16, 16, 20000000, 4), "none"), ((32, 32, 20000000, 4), "none"), ((32, 16, 30720000, 8), "none"),
    ((100, 16, 20000000, 4), "none"), ((128, 32, 20000000, 4), "tall"), ((5000, 17, 25500000, 4), "tall"),
    ((16, 16, 300000, 4), "small"), ((32, 32, 9000000, 4), "small"), ((100, 20, 9000000, 4), "tall"),
    ((100, 20, 9000000, 8), "none"), ((100, 20, 2000000, 8), "tall"), ((20, 20, 4000000, 16), "none"),
    ((20, 16, 300000, 16), "tall"), ((24, 32, 300000, 16), "small"), ((15, 4000, 60000, 4), "none"),
    ((64, 64, 20480000, 4), "small"), ((6000, 5000, 30000000, 4), "large"), ((1000, 700, 700000, 4), "small"),
], ids=str)
def test_binary_transpose_tiles(args, want):
    assert _core._binary_tile(*args) == want


# (slices, axis, columns), element bytes -> kernel of a cumsum down the axis, rows of loads in flight, streaming
@pytest.mark.parametrize("shape,es,want", [
    ((1, 8192, 4096), 4, ("tiles", True)), ((1, 8193, 4099), 4, ("tiles", True)), ((3000, 1000, 24), 4, ("tiles", False)),
    ((10000, 500, 5), 4, (32, False)), ((50000, 500, 2), 4, (32, False)), ((10000, 1000, 3), 8, (32, False)),
    ((1000, 500, 5), 4, ("tiles", False)), ((30000, 100, 7), 4, (32, False)), ((5000, 384, 32), 4, (16, True)),
    ((1, 300, 20000), 4, (32, True)), ((500, 300, 16), 4, (32, False)), ((1, 1000, 131072), 4, (16, True)),
    ((1, 600, 100000), 8, ("none", False)), ((1, 1000, 262144), 4, ("none", False)), ((1, 63, 4096), 4, ("none", False)),
    ((1000, 64, 2), 4, ("none", False)), ((10000, 64, 2), 4, ("none", False)), ((100, 100, 64), 8, (32, True)),
    ((32768, 262144, 2), 4, (32, False)),  # more lanes than a grid dim of tiles holds
], ids=str)
def test_column_scan_routes(shape, es, want):
    o, L, c = shape
    r = _core._route_scan(list(shape), [L * c, c, 1], 1, es)
    assert (r["kind"], r["stream"]) == want if isinstance(want[0], str) else (r["kind"], r["depth"], r["stream"]) == ("lanes",) + want
