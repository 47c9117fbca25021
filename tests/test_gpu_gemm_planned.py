"""fp4_gemm_tiled with the planner's own choice where it changes kind: 32, 33,
64 and 65 rows (few-row kernel and tiles), narrow matrices (several K splits),
ragged rows and columns, one row tile past a full one; every element against
the float64 contraction of the same codes (1e-5 of sum |a w|, the bar of the
tiled kernels' own tests)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LEVELS = np.array([0, .5, 1, 1.5, 2, 3, 4, 6, -0., -.5, -1, -1.5, -2, -3, -4, -6])


def _mx(rng, rows, k):
    codes = rng.integers(0, 256, (rows, k // 2), dtype=np.uint8)
    scales = rng.integers(118, 125, (rows, k // 32), dtype=np.uint8)
    v = np.stack((LEVELS[codes & 15], LEVELS[codes >> 4]), -1).reshape(rows, k // 32, 32)
    return codes, scales, (v * np.exp2(scales.astype(np.float64) - 127)[..., None]).reshape(rows, k)


@pytest.mark.parametrize("m,n,k", [(32, 260, 1024), (33, 260, 1024), (33, 8196, 512), (64, 1024, 8192), (64, 4100, 512),
                                   (65, 1024, 3328), (80, 292, 1024), (129, 516, 2304), (257, 2052, 768), (300, 4356, 512),
                                   (513, 1028, 1792), (700, 260, 1280)])
def test_planned_gemm(rf, stream, m, n, k):
    rng = np.random.default_rng(m + n + k)
    ac, asc, a = _mx(rng, m, k)
    wc, wsc, w = _mx(rng, n, k)
    buf = {}
    for name, c, s, rows in (("a", ac, asc, m), ("w", wc, wsc, n)):
        dc, ds = rf.DeviceBuffer.from_host(c, stream), rf.DeviceBuffer.from_host(s, stream)
        dt = rf.DeviceBuffer.zeroed(rf.mx4_scales_tiled_bytes(rows, k), np.uint8, stream)
        rf.mx4_scales_tile(stream, rows, k, ds, dt)
        buf[name] = (dc, ds, dt)
    out = rf.DeviceBuffer.zeroed(m * n, np.float32, stream)
    for _ in range(2):  # a second call finds the split workspace as the first left it
        rf.fp4_gemm_tiled(stream, m, n, k, *buf["a"], *buf["w"], out)
    got = out.to_host(m * n, np.float32, stream).reshape(m, n)
    bad = abs(got - a @ w.T) > 1e-5 * (abs(a) @ abs(w).T)
    assert not bad.any(), (rf.gemm_plan_kernel(m, n, k), int(bad.sum()))


def test_prefill_epilogue_planned(rf, stream):
    """Where the plain gate|up GEMM is the few-row kernel (narrow matrices to 64
    rows) there is no SwiGLU epilogue; wide or tall ones have it."""
    assert rf.gemm_plan_kernel(64, 4096, 2048).startswith("rfp4_gemm_rows_")
    for m, ffn, k in ((32, 4096, 2048), (64, 2048, 2048), (64, 2048, 1024)):
        assert rf.prefill_epilogue_kernel(m, ffn, k) == ""
    assert rf.prefill_epilogue_kernel(700, 14336, 4096) == "rfp4_gemm_256x256_ppsw"
    assert rf.prefill_epilogue_kernel(128, 5632, 2048).endswith("_sw")
    assert rf.prefill_epilogue_kernel(700, 6144, 4096, 128).endswith("_rope")
    assert rf.prefill_epilogue_kernel(700, 6144, 4096, 96) == ""
