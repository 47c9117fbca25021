"""The few-row GEMM's wide form (a wave per 16 W rows and all of K) against
its K-split form, bit for bit: both start each 512-value segment's products
from zero and add the segments in order."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# n: one partial fragment, a ragged last workgroup, one fragment more than 8
# waves on each of 256 CUs take in a round (two rounds of five waves), three
# rounds; every segment count of 512..4096
@pytest.mark.parametrize("m", [1, 16, 17, 32])
@pytest.mark.parametrize("n,k", [(4, 512), (20, 4096), (1044, 1024), (4100, 1536), (36, 2048), (2052, 2560), (116, 3072),
                                 (12292, 3584), (32772, 512), (36868, 4096), (69636, 1024)])
def test_wide_form_equals_k_split_form(rf, stream, m, n, k):
    rng = np.random.default_rng(m * 131 + n + k)
    dev = []
    for rows in (m, n):
        dev += [rf.DeviceBuffer.from_host(rng.integers(0, 256, rows * k // 2, dtype=np.uint8), stream),
                rf.DeviceBuffer.from_host(rng.integers(118, 128, rows * k // 32, dtype=np.uint8), stream)]
    out = []
    try:
        for nf in (1, 4):
            rf.check(rf.load().rfp4_debug_gemm_plan(5, nf))
            assert rf.gemm_plan(m, n, k) == (16 if m <= 16 else 32, 16 * nf, nf)
            c = rf.DeviceBuffer.from_host(np.full(m * n + 64, np.nan, np.float32), stream)
            rf.fp4_gemm(stream, m, n, k, *dev, c)
            out.append(c.to_host(m * n + 64, np.float32, stream))
    finally:
        rf.check(rf.load().rfp4_debug_gemm_plan(-1, 0))
    assert np.isnan(out[1][m * n:]).all()
    np.testing.assert_array_equal(out[0].view(np.uint32), out[1].view(np.uint32))
