"""GPU parity of arrays large enough for streaming loads (32 MB of input) and stores (32 and 64 MB of output),
which smaller arrays never reach.  Elementwise results and casts are exact."""
import numpy as np
import pytest

import musapy_amd as ms
from tests.conftest import assert_bits_equal
from tests.test_gpu_unaligned import dev, values

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("src,dst", [("int8", "float64"), ("uint8", "float32"), ("int16", "float64"),
                                     ("float32", "float64"), ("float64", "float32")])
def test_casts(src, dst):
    n = (64 << 20) // np.dtype(dst).itemsize
    x = np.random.default_rng(3).integers(-100 if src[0] != "u" else 0, 100, n + 4).astype(src)
    X = dev(x)
    short = {"float64": "f64", "float32": "f32"}[dst]
    for lo, hi in ((0, n), (0, n + 1), (3, n + 4)):
        assert_bits_equal(ms.astype(X[lo:hi], short).numpy(), x[lo:hi].astype(dst), f"{src} -> {dst} [{lo}:{hi}]")
