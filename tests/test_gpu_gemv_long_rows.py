"""GEMV rows of 5, 6 and 8 slices of 2048 values against the slice loop, bit
for bit (each lane adds the same chunks in the same order)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("k", [8224, 10208, 10240, 10272, 12288, 14368, 16352, 16384, 16416])
@pytest.mark.parametrize("n", [1, 7, 2049])
@pytest.mark.parametrize("f32scale,resid", [(False, False), (False, True), (True, False)])
def test_long_rows_equal_slice_loop(rf, stream, n, k, f32scale, resid):
    rng = np.random.default_rng(n + k)
    w = rf.DeviceBuffer.from_host(rng.integers(0, 256, n * k // 2, dtype=np.uint8), stream)
    sc = rng.uniform(0.5, 2, n * k // 32).astype(np.float32) if f32scale else rng.integers(118, 128, n * k // 32, dtype=np.uint8)
    sc = rf.DeviceBuffer.from_host(sc, stream)
    x = rf.DeviceBuffer.from_host(rng.standard_normal(k).astype(np.float32), stream)
    y0 = np.concatenate([rng.standard_normal(n), np.full(8, np.nan)]).astype(np.float32)
    fn = rf.fp4_gemv if f32scale else rf.mx4_gemv_residual if resid else rf.mx4_gemv
    out = []
    try:
        for slices in (-1, 0):
            rf.check(rf.load().rfp4_debug_gemv_variant(0, slices))
            y = rf.DeviceBuffer.from_host(y0, stream)
            fn(stream, n, k, w, sc, x, y)
            out.append(y.to_host(n + 8, np.float32, stream))
    finally:
        rf.check(rf.load().rfp4_debug_gemv_variant(0, -1))
    assert np.isnan(out[0][n:]).all() and np.isfinite(out[0][:n]).all()
    np.testing.assert_array_equal(out[0].view(np.uint32), out[1].view(np.uint32))


@pytest.mark.parametrize("k", [96, 2080, 8224, 10208, 14368])
def test_infinite_last_value(rf, stream, k):
    """An infinite x in the last, partial slice: the lanes past it, which read
    that chunk again, add nothing (a zero factor would make the sums NaN)."""
    n = 9
    w = rf.DeviceBuffer.from_host(np.full(n * k // 2, 0x22, np.uint8), stream)  # every code 1.0
    sc = rf.DeviceBuffer.from_host(np.full(n * k // 32, 127, np.uint8), stream)
    x = np.ones(k, np.float32)
    x[-1] = np.inf
    y = rf.DeviceBuffer.zeroed(n, np.float32, stream)
    rf.mx4_gemv(stream, n, k, w, sc, rf.DeviceBuffer.from_host(x, stream), y)
    np.testing.assert_array_equal(y.to_host(n, np.float32, stream), np.full(n, np.inf, np.float32))
