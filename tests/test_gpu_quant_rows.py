"""mx4_quantize_tiled beyond one pass of its grid (65536 workgroups of 2048
values, then a stride) and from sources at their least alignment: the same
bytes as the rows quantized on their own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("bf16,shift", [(True, 8), (False, 16)])
def test_quantize_past_one_grid_pass(rf, stream, bf16, shift):
    rows, k, tail = 32768 + 40, 4096, 40
    rng = np.random.default_rng(9)
    src = rng.standard_normal((128, k)).astype(np.float32)
    if bf16:
        src = (src.view(np.uint32) >> 16).astype(np.uint16)
    src = np.concatenate([np.zeros(shift, np.uint8), np.tile(src, (rows // 128 + 1, 1))[:rows].view(np.uint8).reshape(-1)])
    d = rf.DeviceBuffer.from_host(src, stream)
    c, s = rf.DeviceBuffer(rows * k // 2), rf.DeviceBuffer(rows * k // 32)
    st = rf.DeviceBuffer.zeroed(rf.mx4_scales_tiled_bytes(rows, k), np.uint8, stream)
    st2 = rf.DeviceBuffer.zeroed(rf.mx4_scales_tiled_bytes(rows, k), np.uint8, stream)
    rf.mx4_quantize_tiled(stream, rows, k, d.ptr + shift, bf16, c, s, st)
    rf.mx4_scales_tile(stream, rows, k, s, st2)
    n = rf.mx4_scales_tiled_bytes(rows, k)
    np.testing.assert_array_equal(st.to_host(n, np.uint8, stream), st2.to_host(n, np.uint8, stream))
    c1, s1 = rf.DeviceBuffer(tail * k // 2), rf.DeviceBuffer(tail * k // 32)
    last = rf.DeviceBuffer.from_host(src[-tail * k * (2 if bf16 else 4):], stream)
    rf.mx4_quantize(stream, tail, k, last, bf16, c1, s1)
    for got, ref, row in ((c, c1, k // 2), (s, s1, k // 32)):
        np.testing.assert_array_equal(got.to_host(rows * row, np.uint8, stream)[-tail * row:], ref.to_host(tail * row, np.uint8, stream))
