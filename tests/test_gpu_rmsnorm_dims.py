"""rmsnorm at the edges of its register forms (2, 4, 8 elements per thread of
1024, then the loop), out of place and in place, f32 and fp16 weights."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dim", [1, 63, 1024, 1025, 2047, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 20000])
@pytest.mark.parametrize("f16", [False, True])
def test_rmsnorm_dims(rf, stream, dim, f16):
    rng = np.random.default_rng(dim)
    x = (3 * rng.standard_normal(dim)).astype(np.float32)
    w = (1 + 0.1 * rng.standard_normal(dim)).astype(np.float16 if f16 else np.float32)
    ref = x.astype(np.float64) / np.sqrt((x.astype(np.float64) ** 2).mean() + 1e-5) * w.astype(np.float64)
    dx, dw = rf.DeviceBuffer.from_host(x, stream), rf.DeviceBuffer.from_host(w.view(np.uint16) if f16 else w, stream)
    y = rf.DeviceBuffer.from_host(np.full(dim + 8, np.nan, np.float32), stream)
    fn = rf.rmsnorm_f16w if f16 else rf.rmsnorm
    fn(stream, dim, 1e-5, dx, dw, y)
    out = y.to_host(dim + 8, np.float32, stream)
    # the mean of squares from per-thread sums of up to 20 terms and two more
    # levels of at most 16: under 40 roundings of 2^-24, halved by the root;
    # five more in the division, root, reciprocal and products
    np.testing.assert_allclose(out[:dim], ref, rtol=25 * 2.0 ** -24, atol=0)
    assert np.isnan(out[dim:]).all()
    fn(stream, dim, 1e-5, dx, dw, dx)
    np.testing.assert_array_equal(dx.to_host(dim, np.float32, stream), out[:dim])
